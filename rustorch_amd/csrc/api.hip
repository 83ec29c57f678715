// C ABI of librt_attn_hip.so (declared in include/rt_attn.h): argument checks in the
// reference's order, device selection, host staging for the slice entry points, kernel dispatch.
// There is no CPU path in this library.
#include <dlfcn.h>
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <exception>
#include <map>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "../../include/rt_attn.h"
#include "rt_kernels.hpp"

#define RT_API extern "C" __attribute__((visibility("default")))

namespace {

void clear_err(rt_err_detail* e) {
    if (e) {
        e->which = -1;
        e->expected = e->got = e->got2 = 0;
        e->hip_error = 0;
        e->message[0] = 0;
    }
}

int fail(rt_err_detail* e, int status, int which, uint64_t expected, uint64_t got, const char* msg, uint64_t got2 = 0) {
    if (e) {
        e->which = which;
        e->expected = expected;
        e->got = got;
        e->got2 = got2;
        e->hip_error = 0;
        snprintf(e->message, sizeof(e->message), "%s", msg ? msg : "");
    }
    return status;
}

int fail_hip(rt_err_detail* e, hipError_t code, const char* where) {
    if (e) {
        e->which = -1;
        e->expected = e->got = e->got2 = 0;
        e->hip_error = (int32_t)code;
        snprintf(e->message, sizeof(e->message), "%s: %s", where, hipGetErrorString(code));
    }
    return RT_ERR_HIP;
}

#define HIP_TRY(expr, where)                                  \
    do {                                                      \
        hipError_t _e = (expr);                               \
        if (_e != hipSuccess) return fail_hip(err, _e, where); \
    } while (0)

// Behind the body of an entry that may allocate on the host: no exception passes a C entry.
#define RT_NO_THROW                                               \
    catch (const std::exception& e) {                             \
        return fail_hip(err, hipErrorOutOfMemory, e.what());      \
    }

int g_num_cus = 0;
int g_decode_waves = 0;  // one-wave workgroups one launch of the decode kernel keeps resident
std::mutex g_init_mutex;
std::atomic<int> g_init_status{-1};  // -1: not tried
char g_init_msg[160];

// Finds a gfx950 device once per process.  Never falls back to anything else.
int ensure_device(rt_err_detail* err, int device = -1) {
    if (device < 0 && g_init_status.load(std::memory_order_acquire) == RT_OK) return RT_OK;  // every call but the first
    std::lock_guard<std::mutex> lock(g_init_mutex);
    if (g_init_status == RT_OK && device < 0) return RT_OK;
    int count = 0;
    hipError_t e = hipGetDeviceCount(&count);
    if (e != hipSuccess || count == 0) {
        (void)hipGetLastError();
        snprintf(g_init_msg, sizeof(g_init_msg), "no HIP device visible (%s)",
                 e == hipSuccess ? "count is 0" : hipGetErrorString(e));
        g_init_status = RT_ERR_NO_DEVICE;
        return fail(err, RT_ERR_NO_DEVICE, -1, 0, 0, g_init_msg);
    }
    int dev = device >= 0 ? device : 0;
    if (device < 0) (void)hipGetDevice(&dev);
    if (dev >= count) {
        snprintf(g_init_msg, sizeof(g_init_msg), "device %d requested, %d visible", dev, count);
        return fail(err, RT_ERR_NO_DEVICE, -1, (uint64_t)count, (uint64_t)dev, g_init_msg);
    }
    hipDeviceProp_t prop;
    e = hipGetDeviceProperties(&prop, dev);
    if (e != hipSuccess) return fail_hip(err, e, "hipGetDeviceProperties");
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
        snprintf(g_init_msg, sizeof(g_init_msg), "device %d is %s; this library holds gfx950 code only", dev,
                 prop.gcnArchName);
        g_init_status = RT_ERR_NO_DEVICE;
        return fail(err, RT_ERR_NO_DEVICE, -1, 0, 0, g_init_msg);
    }
    if (device >= 0) {
        e = hipSetDevice(dev);
        if (e != hipSuccess) return fail_hip(err, e, "hipSetDevice");
    }
    // the decode kernel (one wave, ~18 KB LDS, <= 256 VGPRs) fits 8 times on a CU; one wave per SIMD already
    // streams at the rate the memory system gives, and fewer waves leave fewer partials to merge
    g_num_cus = prop.multiProcessorCount;
    g_decode_waves = prop.multiProcessorCount * 4;
    g_init_status = RT_OK;
    return RT_OK;
}

// validate() of cpu_forward.rs:142-169 followed by Mask::validate (mask.rs:51-65)
int validate_flash(const rt_attention_shape* s, size_t qn, size_t kn, size_t vn, size_t on, int mask_kind,
                   size_t keep_n, rt_err_detail* err) {
    if (s->dim == 0) return fail(err, RT_ERR_ZERO_DIM, -1, 0, 0, "dim must be > 0");
    uint64_t expected = s->batch * s->heads * s->seq * s->dim;
    const size_t lens[3] = {qn, kn, vn};
    static const char* names[3] = {"q", "k", "v"};
    for (int i = 0; i < 3; i++)
        if (lens[i] != expected) {
            char msg[96];
            snprintf(msg, sizeof(msg), "%s buffer has %zu elements, expected %llu", names[i], lens[i],
                     (unsigned long long)expected);
            return fail(err, RT_ERR_BUFFER_SHAPE_MISMATCH, i, expected, lens[i], msg);
        }
    if (on != expected) return fail(err, RT_ERR_OUTPUT_SHAPE_MISMATCH, RT_WHICH_OUT, expected, on, "output buffer length");
    if (mask_kind == RT_MASK_PADDING && keep_n != s->seq)
        return fail(err, RT_ERR_PADDING_LENGTH_MISMATCH, -1, s->seq, keep_n, "padding mask length");
    if (mask_kind != RT_MASK_NONE && mask_kind != RT_MASK_CAUSAL && mask_kind != RT_MASK_PADDING)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, (uint64_t)mask_kind, "unknown mask kind");
    return RT_OK;
}

bool fits_int(uint64_t x) { return x <= 0x7fffffffull; }

int check_flash_dims(const rt_attention_shape* s, uint64_t n_kv_heads, rt_err_detail* err) {
    if (!fits_int(s->batch) || !fits_int(s->heads) || !fits_int(s->seq) || !fits_int(s->dim) || s->batch > 65535 ||
        s->heads > 65535)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, 0, "shape too large for the launch grid");
    if (n_kv_heads == 0 || s->heads % n_kv_heads != 0)
        return fail(err, RT_ERR_HEAD_COUNT_MISMATCH, -1, s->heads, n_kv_heads, "heads not divisible by n_kv_heads");
    return RT_OK;
}

// bnhd: tensors are [batch, seq, heads, dim] instead of [batch, heads, seq, dim]
// rt_set_strict_non_finite_v: off by default
std::atomic<int> g_strict_v{0};

// After a causal forward, when the strict switch is on: the pass that gives query rows the reference's NaN for
// non-finite V elements at keys they do not see (the forward kernels skip those key tiles).
int strict_pass(hipStream_t stream, const rt_attention_shape* s, uint64_t n_kv_heads, const void* v, void* out,
                const int32_t* seq_lens, int mask_kind, bool bnhd, bool bf16, rt_err_detail* err) {
    if (mask_kind != rt::kMaskCausal && mask_kind != rt::kMaskVarlenCausal) return RT_OK;
    if (!g_strict_v.load(std::memory_order_relaxed)) return RT_OK;
    rt::StrictVParams p{};
    p.v = v;
    p.out = out;
    p.seq_lens = seq_lens;
    p.batch = (int)s->batch;
    p.heads = (int)s->heads;
    p.kv_heads = (int)n_kv_heads;
    p.seq = (int)s->seq;
    p.dim = (int)s->dim;
    if (bnhd) {
        p.lo = rt::layout_bnhd((long long)s->heads, (long long)s->seq, p.dim);
        p.lkv = rt::layout_bnhd((long long)n_kv_heads, (long long)s->seq, p.dim);
    } else {
        p.lo = rt::layout_bhnd((long long)s->heads, (long long)s->seq, p.dim);
        p.lkv = rt::layout_bhnd((long long)n_kv_heads, (long long)s->seq, p.dim);
    }
    HIP_TRY(rt::launch_strict_hidden_v(stream, p, bf16), "strict_hidden_v launch");
    return RT_OK;
}

int flash_f32_device(hipStream_t stream, const rt_attention_shape* s, uint64_t n_kv_heads, const float* q,
                     const float* k, const float* v, int mask_kind, const uint8_t* keep, float* out,
                     rt_err_detail* err, bool bnhd = false, const float* bias = nullptr, long long bias_bh_stride = 0,
                     float* lse = nullptr, uint64_t seq_kv = 0) {
    if (s->dim > 512) return fail(err, RT_ERR_UNSUPPORTED, -1, 512, s->dim, "f32 flash kernels cover dim <= 512");
    if (s->dim > 256) {
        // beyond the tiled kernels: one workgroup per query row (any speed), with flash_forward's masks and row rules
        if (s->seq > 0x7fffffffull || seq_kv > 0x7fffffffull) return fail(err, RT_ERR_UNSUPPORTED, -1, 0, 0, "shape too large for the launch grid");
        rt::AttnRowsParams r{};
        r.q = q;
        r.k = k;
        r.v = v;
        r.out = out;
        r.batch = (int)s->batch;
        r.heads = (int)s->heads;
        r.kv_heads = (int)n_kv_heads;
        r.seq_q = (int)s->seq;
        r.kv_len = r.kv_stride = (int)(seq_kv ? seq_kv : s->seq);
        r.dim = (int)s->dim;
        r.head_map = 0;
        r.scale = 1.0f / sqrtf((float)s->dim);
        r.bias = bias;
        r.bias_bh_stride = bias_bh_stride;
        r.use_layout = 1;
        if (bnhd) {
            r.lq = r.lo = rt::layout_bnhd((long long)s->heads, (long long)s->seq, r.dim);
            r.lkv = rt::layout_bnhd((long long)n_kv_heads, (long long)r.kv_len, r.dim);
        } else {
            r.lq = r.lo = rt::layout_bhnd((long long)s->heads, (long long)s->seq, r.dim);
            r.lkv = rt::layout_bhnd((long long)n_kv_heads, (long long)r.kv_len, r.dim);
        }
        r.mask = mask_kind;
        r.keep = keep;
        r.ref_bc = (int)(s->bc == 0 ? 1 : (s->bc > 0x7fffffffull ? 0x7fffffff : s->bc));
        r.flash_rows = 1;
        r.lse = lse;
        HIP_TRY(rt::launch_attn_rows_f32(stream, r), "attn_rows_f32 launch");
        return seq_kv ? RT_OK : strict_pass(stream, s, n_kv_heads, v, out, nullptr, mask_kind, bnhd, false, err);
    }
    rt::FlashF32Params p{};
    p.bias = bias;
    p.bias_bh_stride = bias_bh_stride;
    p.lse = lse;
    p.q = q;
    p.k = k;
    p.v = v;
    p.out = out;
    p.keep = keep;
    p.batch = (int)s->batch;
    p.heads = (int)s->heads;
    p.kv_heads = (int)n_kv_heads;
    p.group = (int)(s->heads / n_kv_heads);
    p.seq = (int)s->seq;
    p.dim = (int)s->dim;
    p.seq_kv = (int)seq_kv;
    p.mask = mask_kind;
    p.ref_bc = (int)(s->bc == 0 ? 1 : (s->bc > 0x7fffffffull ? 0x7fffffff : s->bc));
    p.scale = 1.0f / sqrtf((float)s->dim);
    p.n_cus = g_num_cus;
    const long long kv_rows = (long long)(seq_kv ? seq_kv : s->seq);
    if (bnhd) {
        p.lq = p.lo = rt::layout_bnhd((long long)s->heads, (long long)s->seq, p.dim);
        p.lkv = rt::layout_bnhd((long long)n_kv_heads, kv_rows, p.dim);
    } else {
        p.lq = p.lo = rt::layout_bhnd((long long)s->heads, (long long)s->seq, p.dim);
        p.lkv = rt::layout_bhnd((long long)n_kv_heads, kv_rows, p.dim);
    }
    HIP_TRY(rt::launch_flash_f32(stream, p), "flash_fwd_f32 launch");
    return seq_kv ? RT_OK : strict_pass(stream, s, n_kv_heads, v, out, nullptr, mask_kind, bnhd, false, err);
}

// Scratch the library keeps for entry points whose reference signature has no workspace argument: one buffer per
// (device, stream), allocated on the first call that needs it and kept until rt_stream_destroy / rt_shutdown.
// Calls on one stream are ordered, so they can share it; calls on different streams get different buffers.  When a
// later call needs more, a larger block is allocated and the old one is RETIRED, not freed: another thread may have
// been handed the old pointer and not yet enqueued its kernels (the lock below covers the bookkeeping only, not
// the caller's launches), and kernels already enqueued may still use it.  Retired blocks are freed with the
// stream's entry.  The first call on a stream allocates (hipMalloc): not for use under stream capture.
struct StreamWs {
    void* ptr = nullptr;
    size_t bytes = 0;
    std::vector<void*> retired;
};
std::mutex g_ws_mutex;
std::map<std::pair<int, hipStream_t>, StreamWs> g_ws;

int stream_workspace(hipStream_t stream, size_t bytes, float** out, rt_err_detail* err) {
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev), "hipGetDevice");
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    StreamWs& w = g_ws[{dev, stream}];
    if (w.bytes < bytes) {
        // grow geometrically, so that a context that lengthens token by token retires a handful of blocks at most
        size_t want = std::max<size_t>(std::max<size_t>(bytes, (size_t)1 << 20), 2 * w.bytes);
        w.retired.reserve(w.retired.size() + 1);
        void* fresh = nullptr;
        // (another thread may be capturing its own stream, which an allocation would end with an error)
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        HIP_TRY(hipThreadExchangeStreamCaptureMode(&mode), "hipThreadExchangeStreamCaptureMode");
        const hipError_t got = hipMalloc(&fresh, want);
        (void)hipThreadExchangeStreamCaptureMode(&mode);
        HIP_TRY(got, "hipMalloc workspace");
        if (w.ptr) w.retired.push_back(w.ptr);
        w.ptr = fresh;
        w.bytes = want;
    }
    *out = (float*)w.ptr;
    return RT_OK;
}

// frees what a stream's entry holds; the caller holds g_ws_mutex and has made sure the stream is idle
void release_stream_ws(StreamWs& w) {
    if (w.ptr) (void)hipFree(w.ptr);
    for (void* r : w.retired) (void)hipFree(r);
    w.ptr = nullptr;
    w.bytes = 0;
    w.retired.clear();
}

// Scratch that needs no allocation: the library's second fixed block is cut into rt::kStreamSlots slots, and a
// (device, stream) pair is given one the first time it asks (host bookkeeping only: nothing is allocated, so the
// call may be the first one under stream capture).  A stream keeps its slot until rt_stream_destroy / rt_shutdown;
// when all slots are taken the caller falls back to stream_workspace.
struct SlotTable {
    hipStream_t owner[rt::kStreamSlots] = {};
    bool used[rt::kStreamSlots] = {};
};
std::map<int, SlotTable> g_slots;  // per device; guarded by g_ws_mutex

// The slot of `stream` on the current device (taking a free one if it has none yet), -1 when no slot is free.
int stream_slot(hipStream_t stream, int* slot, rt_err_detail* err) {
    *slot = -1;
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev), "hipGetDevice");
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    SlotTable& t = g_slots[dev];
    for (int i = 0; i < rt::kStreamSlots && *slot < 0; i++)
        if (t.used[i] && t.owner[i] == stream) *slot = i;
    for (int i = 0; i < rt::kStreamSlots && *slot < 0; i++)
        if (!t.used[i]) {
            t.used[i] = true;
            t.owner[i] = stream;
            *slot = i;
        }
    return RT_OK;
}

// A slot's scratch and its size, or *ptr = nullptr when no slot is free.
int stream_slot_scratch(hipStream_t stream, float** ptr, size_t* bytes, rt_err_detail* err) {
    *ptr = nullptr;
    *bytes = 0;
    int slot = -1;
    int rc = stream_slot(stream, &slot, err);
    if (rc || slot < 0) return rc;
    HIP_TRY(rt::stream_static_scratch(slot, ptr, bytes), "hipGetSymbolAddress(stream scratch)");
    return RT_OK;
}

int is_capturing(hipStream_t stream, bool* yes, rt_err_detail* err) {
    *yes = false;
    if (!stream) return RT_OK;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    HIP_TRY(hipStreamIsCapturing(stream, &cap), "hipStreamIsCapturing");
    *yes = cap != hipStreamCaptureStatusNone;
    return RT_OK;
}

// A number no other launch of the process has, its low 8 bits zero.  It starts at no particular place, so that what earlier
// processes left in memory holds no number of this one.
uint64_t next_launch_id() {
    static std::atomic<uint64_t> next{(uint64_t)std::chrono::steady_clock::now().time_since_epoch().count() * 0x9e3779b97f4a7c15ull};
    return next.fetch_add(1, std::memory_order_relaxed) << 8;
}

// How the decode kernels run a call: in the latency form (one launch, partials folded inside it) where that is the faster
// one and the stream is not being captured: a captured launch would bring its id along on every replay, so with more than
// one split a graph gets split and merge kernel, whose two launches cost little inside it.  max_len: the longest context
// there can be.
int plan_decode(hipStream_t stream, rt::DecodeSplitParams& p, int max_len, rt_err_detail* err) {
    const int n_splits = rt::decode_latency_splits(p.batch, p.heads, p.kv_heads, p.dim, p.max_seq, max_len, g_num_cus);
    if (n_splits == 0 || ((uintptr_t)p.out & 7) != 0) return RT_OK;
    if (n_splits > 1) {  // (one split: no partials)
        bool captured = false;
        int rc = is_capturing(stream, &captured, err);
        if (rc || captured) return rc;
        p.launch_id = next_launch_id();
    }
    p.n_splits = n_splits;
    return RT_OK;
}

// hipStreamPerThread is one handle for a stream of every thread, so calls on it share a slot (or block) that nothing
// orders.  They take turns: a call's launch waits, on the GPU, for the event behind the launch of the call before it.
// Under capture, where a wait for work outside it is an error, the call has to do without scratch.
class ScratchTurn {
public:
    int enter(hipStream_t stream, bool* scratch, rt_err_detail* err) {
        *scratch = true;
        if (stream != hipStreamPerThread) return RT_OK;
        bool captured = false;
        int rc = is_capturing(stream, &captured, err);
        if (rc) return rc;
        if (captured) {
            *scratch = false;
            return RT_OK;
        }
        int dev = 0;
        HIP_TRY(hipGetDevice(&dev), "hipGetDevice");
        lock_ = std::unique_lock<std::mutex>(mutex());
        hipEvent_t& e = events()[dev];
        if (!e) HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
        HIP_TRY(hipStreamWaitEvent(stream, e, 0), "hipStreamWaitEvent");
        event_ = e;
        return RT_OK;
    }
    // behind the launch
    int leave(hipStream_t stream, rt_err_detail* err) {
        if (!event_) return RT_OK;
        const hipError_t e = hipEventRecord(event_, stream);
        if (e != hipSuccess) (void)hipStreamSynchronize(stream);
        HIP_TRY(e, "hipEventRecord");
        return RT_OK;
    }
    static void release() {
        std::lock_guard<std::mutex> lock(mutex());
        for (auto& e : events())
            if (e.second) (void)hipEventDestroy(e.second);
        events().clear();
    }

private:
    static std::mutex& mutex() {
        static std::mutex m;
        return m;
    }
    static std::map<int, hipEvent_t>& events() {  // by device
        static std::map<int, hipEvent_t> m;
        return m;
    }
    std::unique_lock<std::mutex> lock_;
    hipEvent_t event_ = nullptr;
};

// the caller holds g_ws_mutex.  Launches of the stream may still use the slot: it is waited for.
void release_stream_slot(int dev, hipStream_t stream) {
    auto it = g_slots.find(dev);
    if (it == g_slots.end()) return;
    for (int i = 0; i < rt::kStreamSlots; i++)
        if (it->second.used[i] && it->second.owner[i] == stream) {
            (void)hipStreamSynchronize(stream);
            it->second.used[i] = false;
        }
}

struct DevPtr {  // a device address inside a Stage's block
    void* p = nullptr;
};

// 16 bytes per thread and round: uploads out of pinned memory, downloads into it
__global__ __launch_bounds__(256) void stage_copy_kernel(uint4* dst, const uint4* src, size_t n16) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (size_t)gridDim.x * blockDim.x) dst[i] = src[i];
}
hipError_t stage_copy(void* dst, const void* src, size_t bytes) {
    hipLaunchKernelGGL(stage_copy_kernel, dim3(64), dim3(256), 0, nullptr, (uint4*)dst, (const uint4*)src, (bytes + 15) / 16);
    return hipGetLastError();
}

// Two threads that help a host-slice call copy: the caller's tensors are as a rule not in its core's cache, and one core
// moves them at about 30 GB/s where the bus takes 55.  A job is a list of copies taken in order by whoever is free, the
// caller included; copy i may start when `ready` > i.  The threads sleep between jobs and end with rt_shutdown.
class CopyCrew {
public:
    struct Piece {
        char* dst;
        const char* src;
        size_t bytes;
    };
    struct Job {
        std::vector<Piece> pieces;
        std::unique_ptr<std::atomic<bool>[]> done;
        std::atomic<size_t> next{0}, ready{0};
        explicit Job(std::vector<Piece> p) : pieces(std::move(p)), done(new std::atomic<bool>[pieces.size()]) {
            for (size_t i = 0; i < pieces.size(); i++) done[i].store(false, std::memory_order_relaxed);
        }
        // takes the next copy if it may start; false: nothing to take
        bool copy_one() {
            size_t i = next.load(std::memory_order_relaxed);
            do {
                if (i >= pieces.size() || ready.load(std::memory_order_acquire) <= i) return false;
            } while (!next.compare_exchange_weak(i, i + 1, std::memory_order_relaxed));
            memcpy(pieces[i].dst, pieces[i].src, pieces[i].bytes);
            done[i].store(true, std::memory_order_release);
            return true;
        }
        void wait(size_t i) {  // for copy i, helping meanwhile
            while (!done[i].load(std::memory_order_acquire))
                if (!copy_one()) __builtin_ia32_pause();
        }
        // copies that have not been taken are not taken any more; returns when those that have been are done
        void close() {
            const size_t taken = next.exchange(pieces.size(), std::memory_order_relaxed);
            for (size_t i = 0; i < std::min(taken, pieces.size()); i++)
                while (!done[i].load(std::memory_order_acquire)) __builtin_ia32_pause();
        }
        bool finished() const { return next.load(std::memory_order_relaxed) >= pieces.size(); }
    };

    // Hands a job to the helpers (one at a time: the caller holds the staging pool, and closes the job when it is through)
    void start(const std::shared_ptr<Job>& job) {
        {
            std::lock_guard<std::mutex> lock(mutex_);
            job_ = job;
            try {
                while (threads_.size() < kHelpers) threads_.emplace_back([this] { help(); });
            } catch (const std::exception&) {  // no thread to be had: the caller copies by itself
            }
        }
        wake_.notify_all();
    }
    void stop() {
        {
            std::lock_guard<std::mutex> lock(mutex_);
            stop_ = true;
        }
        wake_.notify_all();
        for (auto& t : threads_) t.join();
        threads_.clear();
        stop_ = false;
        job_.reset();
    }

private:
    static constexpr size_t kHelpers = 2;
    void help() {
        std::shared_ptr<Job> last;
        for (;;) {
            std::shared_ptr<Job> job;
            {
                std::unique_lock<std::mutex> lock(mutex_);
                wake_.wait(lock, [&] { return stop_ || (job_ && job_ != last); });
                if (stop_) return;
                job = last = job_;
            }
            while (!job->finished())
                if (!job->copy_one()) __builtin_ia32_pause();
        }
    }
    std::mutex mutex_;
    std::condition_variable wake_;
    std::vector<std::thread> threads_;
    std::shared_ptr<Job> job_;
    bool stop_ = false;
};
CopyCrew& crew() {
    static CopyCrew* c = new CopyCrew;  // never destroyed: its threads may sleep in it when the process ends
    return *c;
}

// What the host-slice entries keep between calls: pinned memory (a ring for uploads, a region for results) and, up to
// kStageKeepBytes, the device block of the last call (hipMalloc + hipFree: 23 us per call).  One call at a time holds it.
// Freed by rt_shutdown.
constexpr size_t kStageInBytes = (size_t)16 << 20, kStageOutBytes = (size_t)8 << 20, kStageKeepBytes = (size_t)64 << 20;
constexpr size_t kStageChunk = (size_t)768 << 10;
constexpr size_t kStageDirectBytes = (size_t)512 << 10;  // results up to this size are stored into pinned memory
constexpr size_t kStageCrewBytes = (size_t)8 << 20;  // calls that move this much share their copies with the helpers (16 MiB:
                                                     // 640 -> 550 us; 4 MiB: 171 -> 179, their waking costs more)
constexpr int kStageSlots = 8;
struct StagePool {
    std::mutex mutex;
    char* in = nullptr;
    char* out = nullptr;
    // "the chunk in this slot has landed", by device: an event is recorded in streams of its own device only
    std::map<int, std::array<hipEvent_t, kStageSlots>> landed;
    void* block = nullptr;
    size_t block_bytes = 0;
    int block_dev = -1;

    bool ready(int dev) {  // false: no pinned memory, or no events, to be had
        bool ok = true;
        if (!in)
            ok = hipHostMalloc((void**)&in, kStageInBytes, hipHostMallocPortable) == hipSuccess &&
                 hipHostMalloc((void**)&out, kStageOutBytes, hipHostMallocPortable) == hipSuccess;
        if (ok && !landed.count(dev)) {
            auto& events = landed[dev];
            events.fill(nullptr);
            for (auto& e : events) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
        }
        if (!ok) release();
        return ok;
    }
    void release() {
        if (in) (void)hipHostFree(in);
        if (out) (void)hipHostFree(out);
        for (auto& events : landed)
            for (auto& e : events.second)
                if (e) (void)hipEventDestroy(e);
        landed.clear();
        if (block) (void)hipFree(block);
        in = out = nullptr;
        block = nullptr;
        block_bytes = 0;
        (void)hipGetLastError();
    }
};
StagePool g_stage;

// Staging of one host-slice call: every input, output and scratch buffer of the call sits in ONE device block.
//
// A pageable hipMemcpy costs 60-150 us below a megabyte, and a call has four of them.  Here the inputs go through the
// pinned ring, kStageChunk at a time, each chunk with a copy kernel behind it on the stream, so that the host copies
// one chunk while the GPU fetches the one before (3 MiB: 93 us, against 120 in one piece and 105-125 with DMA copies,
// which cost 10 us each; chunks of 256 KiB 112).  Results come back the same way, the host copying one chunk while the
// next arrives; small ones are written into pinned memory by the attention kernels themselves (larger ones slow the
// kernel down by more than the copy takes: 1 MiB of results 29 -> 47 us).  A call that finds the pool taken (another
// thread is inside a host-slice entry) copies buffer by buffer instead.
class Stage {
public:
    void in(const void* host, size_t bytes, void** dev) { items_.push_back({host, nullptr, bytes, dev, 0, kIn}); }
    // whole_lines: the kernels that write this output store 16 bytes per lane, whole rows
    void out(void* host, size_t bytes, void** dev, bool whole_lines) {
        items_.push_back({nullptr, host, bytes, dev, 0, kOut});
        direct_ = direct_ && whole_lines;
    }
    void scratch(size_t bytes, void** dev) { items_.push_back({nullptr, nullptr, bytes, dev, 0, kScratch}); }

    // Hands out the device pointers and enqueues the uploads (register inputs, then outputs, then scratch).
    int commit(rt_err_detail* err) {
        lock_ = std::unique_lock<std::mutex>(g_stage.mutex, std::try_to_lock);
        HIP_TRY(hipGetDevice(&dev_), "hipGetDevice");
        if (lock_.owns_lock() && !g_stage.ready(dev_)) lock_.unlock();
        size_t in_bytes = 0, out_bytes = 0, total = 0;
        for (auto& it : items_) {
            if (it.kind == kIn) in_bytes += padded(it.bytes);
            if (it.kind == kOut) out_bytes += padded(it.bytes);
        }
        crewed_ = in_bytes + out_bytes >= kStageCrewBytes;
        direct_ = direct_ && lock_.owns_lock() && out_bytes <= kStageDirectBytes;
        size_t out_off = 0;
        for (auto& it : items_) {
            size_t& off = (it.kind == kOut && direct_) ? out_off : total;
            it.off = off;
            off += padded(it.bytes);
        }
        int rc = get_block(total ? total : 256, err);
        if (rc) return rc;
        for (auto& it : items_) *it.dev = ((it.kind == kOut && direct_) ? g_stage.out : block_) + it.off;
        if (!lock_.owns_lock()) {
            for (auto& it : items_)
                if (it.kind == kIn && it.bytes) HIP_TRY(hipMemcpy(*it.dev, it.host_in, it.bytes, hipMemcpyHostToDevice), "copy input");
            return RT_OK;
        }
        // The inputs lie at the head of the block, one behind the other: a copy kernel moves kStageChunk of that range
        // whatever inputs it spans.
        std::vector<CopyCrew::Piece> pieces;
        std::vector<Range> ranges;
        size_t at = 0;  // position in the ring
        for (auto& it : items_) {
            if (it.kind != kIn) continue;
            for (size_t done = 0; done < it.bytes;) {
                if (ranges.empty() || ranges.back().bytes >= kStageChunk) {
                    if (at + kStageChunk + 256 > kStageInBytes) {  // the ring is full: what is in it has to have left
                        rc = upload(pieces, ranges, err);
                        if (rc) return rc;
                        HIP_TRY(hipStreamSynchronize(nullptr), "hipStreamSynchronize");
                        pieces.clear();
                        ranges.clear();
                        at = 0;
                    }
                    ranges.push_back({it.off + done, at, 0, 0});
                }
                Range& r = ranges.back();
                const size_t n = std::min(kStageChunk - r.bytes, it.bytes - done);
                pieces.push_back({g_stage.in + at, (const char*)it.host_in + done, n});
                done += n;
                const size_t step = done == it.bytes ? padded(it.off + done) - (it.off + done - n) : n;  // to where the next input begins
                at += step;
                r.bytes += step;
                r.end_piece = pieces.size();
            }
        }
        return upload(pieces, ranges, err);
    }

    // Brings the outputs back; returns after they are in the caller's buffers.
    int fetch(rt_err_detail* err) {
        if (lock_.owns_lock() && !direct_) {
            // chunk k travels through slot k % kStageSlots
            constexpr size_t kSlotBytes = kStageOutBytes / kStageSlots;
            static_assert(kStageChunk <= kSlotBytes, "a chunk fits its slot");
            std::vector<CopyCrew::Piece> pieces;
            std::vector<const char*> from;
            for (auto& it : items_)
                if (it.kind == kOut)
                    for (size_t done = 0; done < it.bytes; done += kStageChunk) {
                        pieces.push_back({(char*)it.host_out + done, g_stage.out + (pieces.size() % kStageSlots) * kSlotBytes,
                                          std::min(kStageChunk, it.bytes - done)});
                        from.push_back((const char*)*it.dev + done);
                    }
            const size_t n = pieces.size();
            auto& landed = g_stage.landed[dev_];
            std::unique_ptr<Running> run;
            for (size_t sent = 0, got = 0; got < n; got++) {
                for (; sent < n && sent < got + kStageSlots; sent++) {
                    if (run && sent >= kStageSlots) run->job->wait(sent - kStageSlots);
                    HIP_TRY(stage_copy((void*)pieces[sent].src, from[sent], pieces[sent].bytes), "download");
                    HIP_TRY(hipEventRecord(landed[sent % kStageSlots], nullptr), "hipEventRecord");
                }
                HIP_TRY(hipEventSynchronize(landed[got % kStageSlots]), "hipEventSynchronize");
                // the helpers are called when there is something to copy: until then they would spin through the kernel
                if (crewed_ && !run) run.reset(new Running(pieces));
                if (run) run->job->ready.store(got + 1, std::memory_order_release);
                else memcpy(pieces[got].dst, pieces[got].src, pieces[got].bytes);
            }
            for (size_t i = 0; run && i < n; i++) run->job->wait(i);
        } else if (lock_.owns_lock()) {
            HIP_TRY(hipStreamSynchronize(nullptr), "hipStreamSynchronize");
            for (auto& it : items_)
                if (it.kind == kOut && it.bytes) memcpy(it.host_out, *it.dev, it.bytes);
        } else {
            for (auto& it : items_)
                if (it.kind == kOut && it.bytes)
                    HIP_TRY(hipMemcpy(it.host_out, *it.dev, it.bytes, hipMemcpyDeviceToHost), "copy output");
        }
        fetched_ = true;  // the stream has passed everything this call enqueued
        return RT_OK;
    }

    ~Stage() {
        // an early return (a failed launch) may leave work in flight that still uses the block or the pinned memory
        if (block_ && !fetched_) (void)hipStreamSynchronize(nullptr);
        if (own_block_) (void)hipFree(own_block_);
    }

private:
    enum Kind { kIn, kOut, kScratch };
    struct Item {
        const void* host_in;
        void* host_out;
        size_t bytes;
        void** dev;
        size_t off;
        Kind kind;
    };
    static size_t padded(size_t bytes) { return (bytes + 255) & ~(size_t)255; }

    // A list of copies under way, with the helpers where the call is large enough; closed on every way out.
    struct Running {
        std::shared_ptr<CopyCrew::Job> job;
        Running(std::vector<CopyCrew::Piece> pieces) : job(std::make_shared<CopyCrew::Job>(std::move(pieces))) { crew().start(job); }
        ~Running() { job->close(); }
    };

    struct Range {  // of the block and of the ring, with the pieces [.., end_piece) that fill it
        size_t block_off, ring_off, bytes, end_piece;
    };

    // The pieces into the ring, a copy kernel behind each range of it.
    int upload(const std::vector<CopyCrew::Piece>& pieces, const std::vector<Range>& ranges, rt_err_detail* err) {
        std::unique_ptr<Running> run;
        if (crewed_) {
            run.reset(new Running(pieces));
            run->job->ready.store(pieces.size(), std::memory_order_release);
        }
        size_t i = 0;
        for (const Range& r : ranges) {
            for (; i < r.end_piece; i++) {
                if (run) run->job->wait(i);
                else memcpy(pieces[i].dst, pieces[i].src, pieces[i].bytes);
            }
            HIP_TRY(stage_copy(block_ + r.block_off, g_stage.in + r.ring_off, r.bytes), "upload");
        }
        return RT_OK;
    }

    int get_block(size_t bytes, rt_err_detail* err) {
        if (lock_.owns_lock() && bytes <= kStageKeepBytes) {
            if (g_stage.block_bytes < bytes || g_stage.block_dev != dev_) {
                if (g_stage.block) (void)hipFree(g_stage.block);
                g_stage.block = nullptr;
                g_stage.block_bytes = 0;
                const size_t want = std::min(kStageKeepBytes, std::max(bytes + bytes / 2, (size_t)1 << 20));
                HIP_TRY(hipMalloc(&g_stage.block, want), "hipMalloc staging block");
                g_stage.block_bytes = want;
                g_stage.block_dev = dev_;
            }
            block_ = (char*)g_stage.block;
        } else {
            HIP_TRY(hipMalloc(&own_block_, bytes), "hipMalloc staging block");
            block_ = (char*)own_block_;
        }
        return RT_OK;
    }

    std::vector<Item> items_;
    int dev_ = 0;
    char* block_ = nullptr;
    void* own_block_ = nullptr;  // freed with the call; null where the pool's block serves it
    bool direct_ = true;         // results go to pinned memory straight from the kernels
    bool crewed_ = false;        // copies are shared with the helpers
    bool fetched_ = false;
    std::unique_lock<std::mutex> lock_;
};

}  // namespace

RT_API const char* rt_version(void) { return "rt_attn_hip 0.1 (gfx950)"; }

// The file the HIP runtime this library is bound to was loaded from.  A host that wants streams, events or graphs of
// its own must talk to the same runtime instance; a process can hold a second copy (PyTorch wheels ship one), and a
// dlopen by bare name may return that one, whose calls do not know this library's streams.
RT_API const char* rt_hip_runtime_path(void) {
    Dl_info info;
    if (dladdr((void*)&hipGetDeviceCount, &info) && info.dli_fname) return info.dli_fname;
    return "";
}

RT_API const char* rt_status_name(int status) {
    switch (status) {
        case RT_OK: return "Ok";
        case RT_ERR_ZERO_DIM: return "ZeroDim";
        case RT_ERR_BUFFER_SHAPE_MISMATCH: return "BufferShapeMismatch";
        case RT_ERR_OUTPUT_SHAPE_MISMATCH: return "OutputShapeMismatch";
        case RT_ERR_PADDING_LENGTH_MISMATCH: return "PaddingLengthMismatch";
        case RT_ERR_HEAD_COUNT_MISMATCH: return "HeadCountMismatch";
        case RT_ERR_WRONG_INPUT_LEN: return "WrongInputLen";
        case RT_ERR_KV_OVERFLOW: return "Overflow";
        case RT_ERR_KV_WRONG_INPUT_LEN: return "KvWrongInputLen";
        case RT_ERR_ROPE_WRONG_INPUT_LEN: return "RopeWrongInputLen";
        case RT_ERR_ROPE_POSITION_OVERFLOW: return "PositionOverflow";
        case RT_ERR_NULL_POINTER: return "NullPointer";
        case RT_ERR_UNSUPPORTED: return "Unsupported";
        case RT_ERR_WORKSPACE_TOO_SMALL: return "WorkspaceTooSmall";
        case RT_ERR_NO_DEVICE: return "NoDeviceFound";
        case RT_ERR_HIP: return "Driver";
        default: return "Unknown";
    }
}

RT_API int rt_init(int device, rt_err_detail* err) {
    clear_err(err);
    int rc = ensure_device(err, device < 0 ? 0 : device);
    if (rc) return rc;
    // the address of the library's fixed scratch block on this device, looked up here so that the first call of
    // rt_gqa_decode_batched_bf16_noalloc has nothing left to set up
    float* scratch = nullptr;
    size_t scratch_bytes = 0;
    HIP_TRY(rt::decode_static_scratch(&scratch, &scratch_bytes), "hipGetSymbolAddress(static scratch)");
    HIP_TRY(rt::stream_static_scratch(0, &scratch, &scratch_bytes), "hipGetSymbolAddress(stream scratch)");
    return RT_OK;
}

// The f32 kernels that store 16 bytes per lane (the others store single elements, which pinned memory does not take well).
static bool whole_lines_f32(uint64_t dim) { return dim % 4 == 0 && dim <= 128; }

// ---- prefill, host slices -------------------------------------------------------------------------

RT_API int rt_flash_forward_masked_f32(const rt_attention_shape* shape, const float* q, size_t q_len, const float* k,
                                       size_t k_len, const float* v, size_t v_len, int mask_kind,
                                       const uint8_t* keep, size_t keep_len, float* out, size_t out_len,
                                       rt_err_detail* err) try {
    clear_err(err);
    if (!shape) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "shape is NULL");
    int rc = validate_flash(shape, q_len, k_len, v_len, out_len, mask_kind, keep_len, err);
    if (rc) return rc;
    if (shape->seq == 0) return RT_OK;  // cpu_forward.rs:203-206
    size_t n = q_len;
    if (n == 0) return RT_OK;  // batch or heads is 0
    if (!q || !k || !v || !out || (mask_kind == RT_MASK_PADDING && !keep))
        return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    rc = check_flash_dims(shape, shape->heads, err);
    if (rc) return rc;
    rc = ensure_device(err);
    if (rc) return rc;

    Stage st;
    void *dq, *dk, *dv, *dout, *dkeep = nullptr;
    size_t bytes = n * sizeof(float);
    const bool lines = whole_lines_f32(shape->dim);
    st.in(q, bytes, &dq);
    st.in(k, bytes, &dk);
    st.in(v, bytes, &dv);
    if (mask_kind == RT_MASK_PADDING) st.in(keep, keep_len, &dkeep);
    st.out(out, bytes, &dout, lines);
    rc = st.commit(err);
    if (rc) return rc;
    rc = flash_f32_device(nullptr, shape, shape->heads, (const float*)dq, (const float*)dk, (const float*)dv, mask_kind,
                          (const uint8_t*)dkeep, (float*)dout, err);
    if (rc) return rc;
    return st.fetch(err);
} RT_NO_THROW

RT_API int rt_flash_forward_f32(const rt_attention_shape* shape, const float* q, size_t q_len, const float* k,
                                size_t k_len, const float* v, size_t v_len, float* out, size_t out_len,
                                rt_err_detail* err) {
    return rt_flash_forward_masked_f32(shape, q, q_len, k, k_len, v, v_len, RT_MASK_NONE, nullptr, 0, out, out_len,
                                       err);
}

namespace {

// The attention of rt_gqa_forward_f32 on device-resident tensors (arguments already checked).
int gqa_device(hipStream_t stream, const float* q, const float* k, const float* v, float* out, size_t batch,
               size_t n_heads, size_t n_kv_heads, size_t seq_q, size_t seq_kv, size_t head_dim, rt_err_detail* err) {
    auto aligned16 = [](const void* ptr) { return ((uintptr_t)ptr & 15) == 0; };
    if (seq_q == seq_kv) {
        // prefill: unmasked flash; the kernel maps query head -> kv head itself (no replicated copy)
        rt_attention_shape s = {batch, n_heads, seq_q, head_dim, 64, 64};
        return flash_f32_device(stream, &s, n_kv_heads, q, k, v, RT_MASK_NONE, nullptr, out, err);
    }
    if (seq_kv > 0 && head_dim % 4 == 0 && head_dim <= 128 && aligned16(q) && aligned16(k) && aligned16(v) &&
        aligned16(out)) {
        // decode / chunked prefill: every query row attends to all seq_kv keys (gqa.rs:179-208); the tiled kernel
        // with its own key count
        rt_attention_shape s = {batch, n_heads, seq_q, head_dim, 64, 64};
        return flash_f32_device(stream, &s, n_kv_heads, q, k, v, RT_MASK_NONE, nullptr, out, err, false, nullptr, 0,
                                nullptr, seq_kv);
    }
    if (head_dim > 512) return fail(err, RT_ERR_UNSUPPORTED, -1, 512, head_dim, "decode rows kernel covers dim <= 512");
    if (seq_q > 65535 * 32ull) return fail(err, RT_ERR_UNSUPPORTED, -1, 0, seq_q, "seq_q too large");
    rt::AttnRowsParams p{};
    p.q = q;
    p.k = k;
    p.v = v;
    p.out = out;
    p.kv_lens = nullptr;
    p.batch = (int)batch;
    p.heads = (int)n_heads;
    p.kv_heads = (int)n_kv_heads;
    p.seq_q = (int)seq_q;
    p.kv_len = (int)seq_kv;
    p.kv_stride = (int)seq_kv;
    p.dim = (int)head_dim;
    p.head_map = 0;
    p.scale = 1.0f / sqrtf((float)head_dim);
    HIP_TRY(rt::launch_attn_rows_f32(stream, p), "attn_rows_f32 launch");
    return RT_OK;
}

}  // namespace

RT_API int rt_gqa_forward_f32(const float* q, size_t q_len, const float* k, size_t k_len, const float* v,
                              size_t v_len, float* out, size_t out_len, size_t batch, size_t n_heads,
                              size_t n_kv_heads, size_t seq_q, size_t seq_kv, size_t head_dim, rt_err_detail* err) try {
    clear_err(err);
    // gqa.rs:106-141
    if (n_kv_heads == 0 || n_heads % n_kv_heads != 0)
        return fail(err, RT_ERR_HEAD_COUNT_MISMATCH, -1, n_heads, n_kv_heads, "n_heads not divisible by n_kv_heads");
    size_t q_expected = batch * n_heads * seq_q * head_dim;
    size_t kv_expected = batch * n_kv_heads * seq_kv * head_dim;
    if (q_len != q_expected) return fail(err, RT_ERR_WRONG_INPUT_LEN, RT_WHICH_Q, q_expected, q_len, "q length");
    if (k_len != kv_expected) return fail(err, RT_ERR_WRONG_INPUT_LEN, RT_WHICH_K, kv_expected, k_len, "k length");
    if (v_len != kv_expected) return fail(err, RT_ERR_WRONG_INPUT_LEN, RT_WHICH_V, kv_expected, v_len, "v length");
    if (out_len != q_expected) return fail(err, RT_ERR_WRONG_INPUT_LEN, RT_WHICH_OUT, q_expected, out_len, "out length");
    if (seq_q == seq_kv && head_dim == 0)
        // the prefill branch's flash_forward fails with ZeroDim, reported as WrongInputLen{"flash_forward",0,0} (gqa.rs:171-175)
        return fail(err, RT_ERR_WRONG_INPUT_LEN, RT_WHICH_FLASH, 0, 0, "flash_forward");
    if (q_expected == 0) return RT_OK;
    if (!q || !out || (kv_expected && (!k || !v))) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    if (!fits_int(batch) || !fits_int(n_heads) || !fits_int(seq_q) || !fits_int(seq_kv) || !fits_int(head_dim) ||
        batch > 65535 || n_heads > 65535)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, 0, "shape too large for the launch grid");
    int rc = ensure_device(err);
    if (rc) return rc;

    Stage st;
    DevPtr dq, dk, dv, dout;
    st.in(q, q_expected * 4, &dq.p);
    st.in(k, kv_expected * 4, &dk.p);
    st.in(v, kv_expected * 4, &dv.p);
    st.out(out, q_expected * 4, &dout.p, whole_lines_f32(head_dim));
    rc = st.commit(err);
    if (rc) return rc;
    rc = gqa_device(nullptr, (const float*)dq.p, (const float*)dk.p, (const float*)dv.p, (float*)dout.p, batch, n_heads,
                    n_kv_heads, seq_q, seq_kv, head_dim, err);
    if (rc) return rc;
    return st.fetch(err);
} RT_NO_THROW

RT_API int rt_gqa_forward_f32_dev(void* stream, const float* q, const float* k, const float* v, float* out, size_t batch,
                                  size_t n_heads, size_t n_kv_heads, size_t seq_q, size_t seq_kv, size_t head_dim,
                                  rt_err_detail* err) {
    clear_err(err);
    if (n_kv_heads == 0 || n_heads % n_kv_heads != 0)
        return fail(err, RT_ERR_HEAD_COUNT_MISMATCH, -1, n_heads, n_kv_heads, "n_heads not divisible by n_kv_heads");
    if (seq_q == seq_kv && head_dim == 0) return fail(err, RT_ERR_WRONG_INPUT_LEN, RT_WHICH_FLASH, 0, 0, "flash_forward");
    const size_t q_expected = batch * n_heads * seq_q * head_dim, kv_expected = batch * n_kv_heads * seq_kv * head_dim;
    if (q_expected == 0) return RT_OK;
    if (!q || !out || (kv_expected && (!k || !v))) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    if (!fits_int(batch) || !fits_int(n_heads) || !fits_int(seq_q) || !fits_int(seq_kv) || !fits_int(head_dim) ||
        batch > 65535 || n_heads > 65535)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, 0, "shape too large for the launch grid");
    int rc = ensure_device(err);
    if (rc) return rc;
    return gqa_device((hipStream_t)stream, q, k, v, out, batch, n_heads, n_kv_heads, seq_q, seq_kv, head_dim, err);
}

// ---- backward (cpu_backward.rs:46-185) ----------------------------------------------------------------

namespace {

// saved_out / saved_lse non-NULL: the forward is not recomputed and `workspace` holds delta only
int flash_bwd_device(hipStream_t stream, const rt_attention_shape* s, const float* q, const float* k, const float* v,
                     const float* d_out, float* dq, float* dk, float* dv, float* workspace, rt_err_detail* err,
                     const float* saved_out = nullptr, const float* saved_lse = nullptr) {
    if (s->dim > 512) return fail(err, RT_ERR_UNSUPPORTED, -1, 512, s->dim, "f32 backward kernels cover dim <= 512");
    rt::FlashBwdF32Params p{};
    p.q = q;
    p.k = k;
    p.v = v;
    p.d_out = d_out;
    p.dq = dq;
    p.dk = dk;
    p.dv = dv;
    p.batch = (int)s->batch;
    p.heads = (int)s->heads;
    p.seq = (int)s->seq;
    p.dim = (int)s->dim;
    p.scale = 1.0f / sqrtf((float)s->dim);
    p.n_cus = g_num_cus;
    if (saved_out) {
        HIP_TRY(rt::launch_flash_bwd_f32_saved(stream, p, saved_out, saved_lse, workspace), "flash_bwd_f32 launch");
    } else if (s->dim > 256) {
        // the recomputed forward of a head dim the tiled forward kernels do not cover: O and the row statistic from
        // the one-workgroup-per-row kernel, then the backward from them
        const size_t rows = (size_t)(s->batch * s->heads * s->seq);
        float* o = workspace;
        float* lse_ws = workspace + rows * s->dim;
        int rc = flash_f32_device(stream, s, s->heads, q, k, v, RT_MASK_NONE, nullptr, o, err, false, nullptr, 0, lse_ws);
        if (rc) return rc;
        HIP_TRY(rt::launch_flash_bwd_f32_saved(stream, p, o, lse_ws, lse_ws + rows), "flash_bwd_f32 launch");
    } else {
        HIP_TRY(rt::launch_flash_bwd_f32(stream, p, workspace), "flash_bwd_f32 launch");
    }
    return RT_OK;
}

}  // namespace

RT_API size_t rt_flash_backward_workspace_bytes(const rt_attention_shape* shape) {
    if (!shape) return 0;
    if (!fits_int(shape->batch) || !fits_int(shape->heads) || !fits_int(shape->seq) || !fits_int(shape->dim)) return 0;
    return rt::flash_bwd_f32_workspace_floats((int)shape->batch, (int)shape->heads, (int)shape->seq, (int)shape->dim) *
           sizeof(float);
}

RT_API int rt_flash_backward_f32(const rt_attention_shape* shape, const float* q, size_t q_len, const float* k,
                                 size_t k_len, const float* v, size_t v_len, const float* d_out, size_t d_out_len,
                                 float* dq, size_t dq_len, float* dk, size_t dk_len, float* dv, size_t dv_len,
                                 rt_err_detail* err) try {
    clear_err(err);
    if (!shape) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "shape is NULL");
    // cpu_backward.rs:59-74: no ZeroDim check here, unlike the forward
    const uint64_t expected = shape->batch * shape->heads * shape->seq * shape->dim;
    const size_t lens[4] = {q_len, k_len, v_len, d_out_len};
    static const char* names[4] = {"q", "k", "v", "do"};
    static const int which[4] = {RT_WHICH_Q, RT_WHICH_K, RT_WHICH_V, RT_WHICH_DO};
    for (int i = 0; i < 4; i++)
        if (lens[i] != expected) {
            char msg[96];
            snprintf(msg, sizeof(msg), "%s buffer has %zu elements, expected %llu", names[i], lens[i],
                     (unsigned long long)expected);
            return fail(err, RT_ERR_BUFFER_SHAPE_MISMATCH, which[i], expected, lens[i], msg);
        }
    if (dq_len != expected || dk_len != expected || dv_len != expected) {
        size_t got = dq_len > dk_len ? dq_len : dk_len;
        if (dv_len > got) got = dv_len;
        return fail(err, RT_ERR_OUTPUT_SHAPE_MISMATCH, RT_WHICH_OUT, expected, got, "gradient buffer length");
    }
    if (shape->seq == 0 || expected == 0) return RT_OK;
    if (!q || !k || !v || !d_out || !dq || !dk || !dv) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    int rc = check_flash_dims(shape, shape->heads, err);
    if (rc) return rc;
    rc = ensure_device(err);
    if (rc) return rc;

    const size_t bytes = (size_t)expected * sizeof(float);
    Stage st;
    DevPtr in[4], out[3], ws;
    const float* host_in[4] = {q, k, v, d_out};
    float* host_out[3] = {dq, dk, dv};
    for (int i = 0; i < 4; i++) st.in(host_in[i], bytes, &in[i].p);
    for (int i = 0; i < 3; i++) st.out(host_out[i], bytes, &out[i].p, whole_lines_f32(shape->dim));
    st.scratch(rt_flash_backward_workspace_bytes(shape), &ws.p);
    rc = st.commit(err);
    if (rc) return rc;
    rc = flash_bwd_device(nullptr, shape, (const float*)in[0].p, (const float*)in[1].p, (const float*)in[2].p,
                          (const float*)in[3].p, (float*)out[0].p, (float*)out[1].p, (float*)out[2].p, (float*)ws.p, err);
    if (rc) return rc;
    return st.fetch(err);
} RT_NO_THROW

RT_API int rt_flash_backward_f32_dev(void* stream, const rt_attention_shape* shape, const float* q, const float* k,
                                     const float* v, const float* d_out, float* dq, float* dk, float* dv,
                                     void* workspace, size_t workspace_bytes, rt_err_detail* err) {
    clear_err(err);
    if (!shape) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "shape is NULL");
    if (shape->seq == 0 || shape->batch == 0 || shape->heads == 0 || shape->dim == 0) return RT_OK;
    int rc = check_flash_dims(shape, shape->heads, err);
    if (rc) return rc;
    if (!q || !k || !v || !d_out || !dq || !dk || !dv || !workspace)
        return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    const size_t need = rt_flash_backward_workspace_bytes(shape);
    if (workspace_bytes < need || ((uintptr_t)workspace & 15))
        return fail(err, RT_ERR_WORKSPACE_TOO_SMALL, -1, need, workspace_bytes, "backward workspace");
    rc = ensure_device(err);
    if (rc) return rc;
    return flash_bwd_device((hipStream_t)stream, shape, q, k, v, d_out, dq, dk, dv, (float*)workspace, err);
}

RT_API int rt_flash_forward_stats_f32_dev(void* stream, const rt_attention_shape* shape, const float* q, const float* k,
                                          const float* v, float* out, float* lse, rt_err_detail* err) {
    clear_err(err);
    if (!shape) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "shape is NULL");
    if (shape->dim == 0) return fail(err, RT_ERR_ZERO_DIM, -1, 0, 0, "dim must be > 0");
    if (shape->seq == 0 || shape->batch == 0 || shape->heads == 0) return RT_OK;
    int rc = check_flash_dims(shape, shape->heads, err);
    if (rc) return rc;
    if (!q || !k || !v || !out || !lse) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    rc = ensure_device(err);
    if (rc) return rc;
    return flash_f32_device((hipStream_t)stream, shape, shape->heads, q, k, v, RT_MASK_NONE, nullptr, out, err, false,
                            nullptr, 0, lse);
}

RT_API int rt_flash_backward_saved_f32_dev(void* stream, const rt_attention_shape* shape, const float* q, const float* k,
                                           const float* v, const float* out, const float* lse, const float* d_out,
                                           float* dq, float* dk, float* dv, void* workspace, size_t workspace_bytes,
                                           rt_err_detail* err) {
    clear_err(err);
    if (!shape) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "shape is NULL");
    if (shape->seq == 0 || shape->batch == 0 || shape->heads == 0 || shape->dim == 0) return RT_OK;
    int rc = check_flash_dims(shape, shape->heads, err);
    if (rc) return rc;
    if (!q || !k || !v || !out || !lse || !d_out || !dq || !dk || !dv || !workspace)
        return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    const size_t need = (size_t)(shape->batch * shape->heads * shape->seq) * sizeof(float);
    if (workspace_bytes < need)
        return fail(err, RT_ERR_WORKSPACE_TOO_SMALL, -1, need, workspace_bytes, "backward workspace (delta)");
    rc = ensure_device(err);
    if (rc) return rc;
    return flash_bwd_device((hipStream_t)stream, shape, q, k, v, d_out, dq, dk, dv, (float*)workspace, err, out, lse);
}

// ---- prefill, device pointers -----------------------------------------------------------------------

RT_API int rt_flash_forward_f32_dev(void* stream, const rt_attention_shape* shape, uint64_t n_kv_heads,
                                    const float* q, const float* k, const float* v, int mask_kind,
                                    const uint8_t* keep, float* out, rt_err_detail* err) {
    clear_err(err);
    if (!shape) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "shape is NULL");
    if (shape->dim == 0) return fail(err, RT_ERR_ZERO_DIM, -1, 0, 0, "dim must be > 0");
    if (mask_kind < RT_MASK_NONE || mask_kind > RT_MASK_PADDING)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, (uint64_t)mask_kind, "unknown mask kind");
    if (n_kv_heads == 0) n_kv_heads = shape->heads;
    if (shape->seq == 0 || shape->batch == 0 || shape->heads == 0) return RT_OK;
    int rc = check_flash_dims(shape, n_kv_heads, err);
    if (rc) return rc;
    if (!q || !k || !v || !out || (mask_kind == RT_MASK_PADDING && !keep))
        return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    rc = ensure_device(err);
    if (rc) return rc;
    return flash_f32_device((hipStream_t)stream, shape, n_kv_heads, q, k, v, mask_kind, keep, out, err);
}

// Which bf16 prefill kernel serves a call.  RT_ATTN_BF16_PREFILL=tile|persistent|wide in the environment forces one
// where it applies (for measurements and tests); otherwise flash_bf16_common weighs the persistent 8-wave kernel
// against the 4-wave tile kernel.
enum class PrefillKernel { kAuto, kTile, kPersistent, kWide };
// A debug switch for measurements and tests, not part of the reference's surface: rt_debug_force_bf16_prefill_kernel
// sets it; until that is called, the value is what RT_ATTN_BF16_PREFILL=tile|persistent held when the library made its
// first bf16 prefill call (read once: a later change of the environment does not change which kernel a caller gets).
static PrefillKernel parse_prefill_kernel(const char* e) {
    if (!e) return PrefillKernel::kAuto;
    if (strcmp(e, "tile") == 0) return PrefillKernel::kTile;
    if (strcmp(e, "persistent") == 0) return PrefillKernel::kPersistent;
    if (strcmp(e, "wide") == 0) return PrefillKernel::kWide;
    return PrefillKernel::kAuto;
}
static std::atomic<int> g_prefill_forced{-1};  // -1: not set through the API
static PrefillKernel prefill_kernel_override() {
    const int f = g_prefill_forced.load(std::memory_order_relaxed);
    if (f >= 0) return (PrefillKernel)f;
    static const PrefillKernel once = parse_prefill_kernel(getenv("RT_ATTN_BF16_PREFILL"));
    return once;
}
RT_API int rt_debug_force_bf16_prefill_kernel(int which) {
    if (which < 0 || which > 3) return RT_ERR_UNSUPPORTED;
    g_prefill_forced.store(which, std::memory_order_relaxed);
    return RT_OK;
}

RT_API int rt_debug_f32_split_products(const rt_attention_shape* shape, uint64_t seq_kv, int mask_kind, int with_lse) {
    if (!shape || !fits_int(shape->batch) || !fits_int(shape->heads) || !fits_int(shape->seq) || !fits_int(seq_kv) || shape->dim == 0 || shape->dim > 512) return 0;
    rt::FlashF32Params p{};
    p.batch = (int)shape->batch;
    p.heads = (int)shape->heads;
    p.seq = (int)shape->seq;
    p.seq_kv = (int)seq_kv;
    p.dim = (int)shape->dim;
    p.mask = mask_kind;
    p.n_cus = g_num_cus;
    return rt::flash_f32_takes_split(p, with_lse != 0) ? 1 : 0;
}

RT_API int rt_debug_f32_wide_gradients(const rt_attention_shape* shape) {
    if (!shape || !fits_int(shape->batch) || !fits_int(shape->heads) || !fits_int(shape->seq) || shape->dim == 0 || shape->dim > 512) return 0;
    rt::FlashF32Params p{};
    p.batch = (int)shape->batch;
    p.heads = (int)shape->heads;
    p.seq = (int)shape->seq;
    p.dim = (int)shape->dim;
    p.mask = rt::kMaskNone;
    p.n_cus = g_num_cus;
    return rt::flash_f32_gradients_wide(p) ? 1 : 0;
}

RT_API int rt_set_strict_non_finite_v(int on) { return g_strict_v.exchange(on ? 1 : 0); }

static int flash_bf16_common(void* stream, const rt_attention_shape* shape, uint64_t n_kv_heads, const void* q,
                             const void* k, const void* v, int mask, const uint8_t* keep, const int32_t* seq_lens,
                             int zero_padded_rows, void* out, rt_err_detail* err, bool bnhd = false) {
    clear_err(err);
    if (!shape) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "shape is NULL");
    if (shape->dim == 0) return fail(err, RT_ERR_ZERO_DIM, -1, 0, 0, "dim must be > 0");
    if (n_kv_heads == 0) n_kv_heads = shape->heads;
    if (shape->seq == 0 || shape->batch == 0 || shape->heads == 0) return RT_OK;
    int rc = check_flash_dims(shape, n_kv_heads, err);
    if (rc) return rc;
    if (shape->dim > 512)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 512, shape->dim, "bf16 flash kernels cover head dims up to 512");
    // the tile kernel's grid is (heads, batch, query tiles of 128 rows), each dimension below 2^16
    if (shape->heads > 65535 || shape->batch > 65535 || (shape->seq + 127) / 128 > 65535)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, 0, "shape too large for the launch grid");
    if (!q || !k || !v || !out || (mask == rt::kMaskPadding && !keep) || (mask == rt::kMaskVarlenCausal && !seq_lens))
        return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    rc = ensure_device(err);
    if (rc) return rc;
    // The matrix-core kernels move 16 bytes at a time: head dims up to 256 that are a multiple of 8, tensors 16-byte
    // aligned.  Everything else (the reference takes any dim != 0, cpu_forward.rs:142-169) goes to the
    // one-workgroup-per-row kernel: same masks, same row rules, any speed.
    // (so does a K/V slab of 4 GiB or more per (batch, kv head): the tile kernel addresses it with 32-bit offsets)
    const bool tile_addressable = rt::flash_tile_bf16_addressable((long long)shape->seq, (long long)((bnhd ? n_kv_heads : 1) * shape->dim));
    if (shape->dim > 256 || shape->dim % 8 != 0 || (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15) != 0 ||
        !tile_addressable) {
        rt::AttnRowsParams r{};
        r.q = q;
        r.k = k;
        r.v = v;
        r.out = out;
        r.kv_lens = mask == rt::kMaskVarlenCausal ? seq_lens : nullptr;
        r.q_lens = r.kv_lens;
        r.batch = (int)shape->batch;
        r.heads = (int)shape->heads;
        r.kv_heads = (int)n_kv_heads;
        r.seq_q = r.kv_len = r.kv_stride = (int)shape->seq;
        r.dim = (int)shape->dim;
        r.head_map = 0;
        r.scale = 1.0f / sqrtf((float)shape->dim);
        r.use_layout = 1;
        if (bnhd) {
            r.lq = r.lo = rt::layout_bnhd((long long)shape->heads, (long long)shape->seq, r.dim);
            r.lkv = rt::layout_bnhd((long long)n_kv_heads, (long long)shape->seq, r.dim);
        } else {
            r.lq = r.lo = rt::layout_bhnd((long long)shape->heads, (long long)shape->seq, r.dim);
            r.lkv = rt::layout_bhnd((long long)n_kv_heads, (long long)shape->seq, r.dim);
        }
        r.mask = mask == rt::kMaskVarlenCausal ? rt::kMaskCausal : mask;
        r.keep = keep;
        r.ref_bc = (int)(shape->bc == 0 ? 1 : (shape->bc > 0x7fffffffull ? 0x7fffffff : shape->bc));
        r.flash_rows = 1;
        r.zero_padded_rows = zero_padded_rows;
        HIP_TRY(rt::launch_attn_rows_bf16((hipStream_t)stream, r), "attn_rows_bf16 launch");
        return strict_pass((hipStream_t)stream, shape, n_kv_heads, v, out, seq_lens, mask, bnhd, true, err);
    }
    // The persistent kernel needs a job (256 query rows of one head) for every CU and long rows; it multiplies faster than
    // the tile kernel, which balances better: 128-row workgroups that the dispatcher hands out, against whole jobs dealt
    // beforehand.  Head dim 64 is the tile kernel's on every shape tried (N = 700 .. 32768, 3-26 %), and so is a padded
    // batch, a set of jobs of very different lengths.  At head dim 128 the two are weighed by what their busiest worker
    // has to do: a persistent step (256 rows x 128 keys) takes 3.15 us, four tile steps (128 rows x 64 keys) 3.85 us, and
    // either kernel two and a half steps around every job.  (us, persistent / tile, causal, 32 / 8 heads: 2 sequences of
    // 1100 32.6 / 31.1, 1501 45.5 / 46.8, 2048 70.5 / 74.9, 2500 112.8 / 109.9; 1 of 2048 48.4 / 43.8, 4096 124 / 136.)
    // Under a key-padding mask the tile kernel takes another fifth longer and the persistent one stays ahead.
    rt::FlashBf16Params p{};
    p.batch = (int)shape->batch;
    p.heads = (int)shape->heads;
    p.kv_heads = (int)n_kv_heads;
    p.group = (int)(shape->heads / n_kv_heads);
    p.seq = (int)shape->seq;
    p.dim = (int)shape->dim;
    p.mask = mask;
    p.n_workers = g_num_cus;
    const uint64_t jobs256 = (shape->seq + 255) / 256 * shape->batch * shape->heads;
    bool persistent = shape->dim == 128 && shape->seq >= 512 && jobs256 >= (uint64_t)g_num_cus && mask != rt::kMaskVarlenCausal;
    const PrefillKernel forced = prefill_kernel_override();
    if (forced == PrefillKernel::kTile || forced == PrefillKernel::kWide) persistent = false;
    if (forced == PrefillKernel::kPersistent && shape->dim == 128 && mask != rt::kMaskVarlenCausal) persistent = true;
    if (mask == rt::kMaskPadding && shape->seq > (uint64_t)rt::kFlashBf16MaxPaddingKeys) persistent = false;
    if (persistent) {  // that kernel addresses the rows of one (batch, head) slab with 32-bit byte offsets
        const uint64_t pitch_b = (bnhd ? shape->heads : 1) * shape->dim * 2;
        if (shape->seq * pitch_b >= (1ull << 32)) persistent = false;
    }
    if (persistent) {
        const float busiest = rt::plan_flash_bf16(p);
        if (forced == PrefillKernel::kAuto && mask != rt::kMaskPadding) {
            const float tiles = (float)((shape->seq + 127) / 128);  // of 128 rows, each 64 keys a step
            const float steps = tiles * ((mask == rt::kMaskCausal ? tiles + 1.0f : 2.0f * tiles) + 2.5f) * (float)(shape->batch * shape->heads);
            if (3.85f * steps / (4.0f * (float)g_num_cus) + 2.0f < 3.15f * busiest) persistent = false;
        }
    }
    const int dim = (int)shape->dim;
    rt::TensorLayout lq, lkv;
    if (bnhd) {
        lq = rt::layout_bnhd((long long)shape->heads, (long long)shape->seq, dim);
        lkv = rt::layout_bnhd((long long)n_kv_heads, (long long)shape->seq, dim);
    } else {
        lq = rt::layout_bhnd((long long)shape->heads, (long long)shape->seq, dim);
        lkv = rt::layout_bhnd((long long)n_kv_heads, (long long)shape->seq, dim);
    }
    const int ref_bc = (int)(shape->bc == 0 ? 1 : (shape->bc > 0x7fffffffull ? 0x7fffffff : shape->bc));
    const float scale = 1.0f / sqrtf((float)shape->dim);
    if (!persistent) {
        rt::FlashTileParams t{};
        t.q = (const uint16_t*)q;
        t.k = (const uint16_t*)k;
        t.v = (const uint16_t*)v;
        t.out = (uint16_t*)out;
        t.keep = keep;
        // a padded batch: sequence b has seq_lens[b] query positions and as many keys, masked causally
        t.q_lens = mask == rt::kMaskVarlenCausal ? seq_lens : nullptr;
        t.kv_lens = t.q_lens;
        t.batch = (int)shape->batch;
        t.heads = (int)shape->heads;
        t.kv_heads = (int)n_kv_heads;
        t.group = (int)(shape->heads / n_kv_heads);
        t.pack = 1;
        t.n_cus = g_num_cus;
        t.seq_q = t.seq_kv = (int)shape->seq;
        t.dim = dim;
        t.mask = mask == rt::kMaskVarlenCausal ? rt::kMaskCausal : mask;
        t.ref_bc = ref_bc;
        t.zero_padded_rows = zero_padded_rows;
        t.scale = scale;
        t.scale_log2e = scale * rt::kLog2eHost;
        t.lq = t.lo = lq;
        t.lkv = lkv;
        if (forced == PrefillKernel::kWide && rt::flash_wide_bf16_supported(t)) {
            HIP_TRY(rt::launch_flash_wide_bf16((hipStream_t)stream, t), "flash_wide_bf16 launch");
            return strict_pass((hipStream_t)stream, shape, n_kv_heads, v, out, seq_lens, mask, bnhd, true, err);
        }
        HIP_TRY(rt::launch_flash_tile_bf16((hipStream_t)stream, t), "flash_tile_bf16 launch");
        return strict_pass((hipStream_t)stream, shape, n_kv_heads, v, out, seq_lens, mask, bnhd, true, err);
    }
    p.q = (const uint16_t*)q;
    p.k = (const uint16_t*)k;
    p.v = (const uint16_t*)v;
    p.out = (uint16_t*)out;
    p.keep = keep;
    p.ref_bc = ref_bc;
    p.scale_log2e = scale * rt::kLog2eHost;
    p.lq = p.lo = lq;
    p.lkv = lkv;
    HIP_TRY(rt::launch_flash_bf16((hipStream_t)stream, p), "flash_fwd_bf16 launch");
    return strict_pass((hipStream_t)stream, shape, n_kv_heads, v, out, seq_lens, mask, bnhd, true, err);
}

RT_API int rt_flash_forward_bf16_dev(void* stream, const rt_attention_shape* shape, uint64_t n_kv_heads,
                                     const void* q, const void* k, const void* v, int mask_kind, const uint8_t* keep,
                                     void* out, rt_err_detail* err) {
    if (mask_kind < RT_MASK_NONE || mask_kind > RT_MASK_PADDING) {
        clear_err(err);
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, (uint64_t)mask_kind, "unknown mask kind");
    }
    return flash_bf16_common(stream, shape, n_kv_heads, q, k, v, mask_kind, keep, nullptr, 0, out, err);
}

RT_API int rt_flash_forward_bnhd_bf16_dev(void* stream, const rt_attention_shape* shape, uint64_t n_kv_heads,
                                          const void* q, const void* k, const void* v, int mask_kind,
                                          const uint8_t* keep, void* out, rt_err_detail* err) {
    if (mask_kind < RT_MASK_NONE || mask_kind > RT_MASK_PADDING) {
        clear_err(err);
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, (uint64_t)mask_kind, "unknown mask kind");
    }
    return flash_bf16_common(stream, shape, n_kv_heads, q, k, v, mask_kind, keep, nullptr, 0, out, err, true);
}

RT_API int rt_flash_forward_bnhd_f32_dev(void* stream, const rt_attention_shape* shape, uint64_t n_kv_heads,
                                         const float* q, const float* k, const float* v, int mask_kind,
                                         const uint8_t* keep, float* out, rt_err_detail* err) {
    clear_err(err);
    if (!shape) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "shape is NULL");
    if (shape->dim == 0) return fail(err, RT_ERR_ZERO_DIM, -1, 0, 0, "dim must be > 0");
    if (mask_kind < RT_MASK_NONE || mask_kind > RT_MASK_PADDING)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, (uint64_t)mask_kind, "unknown mask kind");
    if (n_kv_heads == 0) n_kv_heads = shape->heads;
    if (shape->seq == 0 || shape->batch == 0 || shape->heads == 0) return RT_OK;
    int rc = check_flash_dims(shape, n_kv_heads, err);
    if (rc) return rc;
    if (!q || !k || !v || !out || (mask_kind == RT_MASK_PADDING && !keep))
        return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    rc = ensure_device(err);
    if (rc) return rc;
    return flash_f32_device((hipStream_t)stream, shape, n_kv_heads, q, k, v, mask_kind, keep, out, err, true);
}

RT_API int rt_mha_flash_forward_f32(const float* q, size_t q_len, const float* k, size_t k_len, const float* v,
                                    size_t v_len, float* out, size_t out_len, size_t batch, size_t seq, size_t heads,
                                    size_t head_dim, rt_err_detail* err) try {
    clear_err(err);
    // the reference transposes to [B,H,T,hd] and calls flash_forward (attention.rs:474-483): same checks, same order
    rt_attention_shape shape = {batch, heads, seq, head_dim, 64, 64};
    int rc = validate_flash(&shape, q_len, k_len, v_len, out_len, RT_MASK_NONE, 0, err);
    if (rc) return rc;
    if (seq == 0 || q_len == 0) return RT_OK;
    if (!q || !k || !v || !out) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    rc = check_flash_dims(&shape, heads, err);
    if (rc) return rc;
    rc = ensure_device(err);
    if (rc) return rc;
    Stage st;
    DevPtr dq, dk, dv, dout;
    size_t bytes = q_len * sizeof(float);
    st.in(q, bytes, &dq.p);
    st.in(k, bytes, &dk.p);
    st.in(v, bytes, &dv.p);
    st.out(out, bytes, &dout.p, whole_lines_f32(head_dim));
    rc = st.commit(err);
    if (rc) return rc;
    rc = flash_f32_device(nullptr, &shape, heads, (const float*)dq.p, (const float*)dk.p, (const float*)dv.p,
                          RT_MASK_NONE, nullptr, (float*)dout.p, err, true);
    if (rc) return rc;
    return st.fetch(err);
} RT_NO_THROW

namespace {

// The attention of rt_mha_forward_masked_f32 on device-resident tensors (arguments already checked).
int mha_masked_device(hipStream_t stream, const float* q, const float* k, const float* v, const float* mask,
                      size_t mask_len, float* out, size_t batch, size_t t_q, size_t t_kv, size_t heads,
                      size_t head_dim, rt_err_detail* err) {
    const size_t one_mask = t_q * t_kv, all_masks = batch * heads * one_mask;
    int rc = RT_OK;
    const long long bias_bh_stride = (mask_len == all_masks && all_masks != one_mask) ? (long long)one_mask : 0;
    auto aligned16 = [](const void* ptr) { return ((uintptr_t)ptr & 15) == 0; };
    if (t_kv > 0 && head_dim % 4 == 0 && head_dim <= 128 && fits_int(t_kv) && aligned16(q) && aligned16(k) &&
        aligned16(v) && aligned16(out)) {
        // a head dim the tiled f32 kernel covers (and 16-byte aligned tensors): the same kernel as the unmasked path,
        // with the mask's row added to the scaled scores and, for cross-attention, its own number of keys
        rt_attention_shape shape = {batch, heads, t_q, head_dim, 64, 64};
        rc = flash_f32_device(stream, &shape, heads, q, k, v, RT_MASK_NONE, nullptr, out, err, true,
                              mask_len ? mask : nullptr, bias_bh_stride, nullptr, t_kv);
        return rc;
    }
    rt::AttnRowsParams p{};
    p.q = q;
    p.k = k;
    p.v = v;
    p.out = out;
    p.kv_lens = nullptr;
    p.batch = (int)batch;
    p.heads = (int)heads;
    p.kv_heads = (int)heads;
    p.seq_q = (int)t_q;
    p.kv_len = (int)t_kv;
    p.kv_stride = (int)t_kv;
    p.dim = (int)head_dim;
    p.head_map = 0;
    p.scale = 1.0f / sqrtf((float)head_dim);
    p.bias = mask_len ? mask : nullptr;
    p.bias_bh_stride = bias_bh_stride;
    p.use_layout = 1;
    p.lq = p.lo = rt::layout_bnhd((long long)heads, (long long)t_q, (int)head_dim);
    p.lkv = rt::layout_bnhd((long long)heads, (long long)t_kv, (int)head_dim);
    HIP_TRY(rt::launch_attn_rows_f32(stream, p), "attn_rows_f32 launch");
    return RT_OK;
}

}  // namespace

RT_API int rt_mha_forward_masked_f32(const float* q, size_t q_len, const float* k, size_t k_len, const float* v,
                                     size_t v_len, const float* mask, size_t mask_len, float* out, size_t out_len,
                                     size_t batch, size_t t_q, size_t t_kv, size_t heads, size_t head_dim,
                                     rt_err_detail* err) try {
    clear_err(err);
    if (head_dim == 0) return fail(err, RT_ERR_ZERO_DIM, -1, 0, 0, "dim must be > 0");
    const size_t embed = heads * head_dim;
    const size_t q_expected = batch * t_q * embed, kv_expected = batch * t_kv * embed;
    if (q_len != q_expected) return fail(err, RT_ERR_BUFFER_SHAPE_MISMATCH, RT_WHICH_Q, q_expected, q_len, "q length");
    if (k_len != kv_expected) return fail(err, RT_ERR_BUFFER_SHAPE_MISMATCH, RT_WHICH_K, kv_expected, k_len, "k length");
    if (v_len != kv_expected) return fail(err, RT_ERR_BUFFER_SHAPE_MISMATCH, RT_WHICH_V, kv_expected, v_len, "v length");
    if (out_len != q_expected) return fail(err, RT_ERR_OUTPUT_SHAPE_MISMATCH, -1, q_expected, out_len, "out length");
    const size_t one_mask = t_q * t_kv, all_masks = batch * heads * one_mask;
    if (!mask) mask_len = 0;
    if (mask_len != 0 && mask_len != one_mask && mask_len != all_masks)
        return fail(err, RT_ERR_WRONG_INPUT_LEN, RT_WHICH_MASK, one_mask, mask_len, "mask length");
    if (q_expected == 0) return RT_OK;
    if (!q || !out || (kv_expected && (!k || !v))) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    if (head_dim > 512) return fail(err, RT_ERR_UNSUPPORTED, -1, 512, head_dim, "rows kernel covers dim <= 512");
    if (heads > 65535 || batch > 65535 || t_q > 0x7fffffffull || t_kv > 0x7fffffffull || embed > 0x7fffffffull)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, 0, "shape too large for the launch grid");
    int rc = ensure_device(err);
    if (rc) return rc;
    Stage st;
    DevPtr dq, dk, dv, dm, dout;
    st.in(q, q_expected * 4, &dq.p);
    st.in(k, kv_expected * 4, &dk.p);
    st.in(v, kv_expected * 4, &dv.p);
    st.in(mask, mask_len * 4, &dm.p);
    st.out(out, q_expected * 4, &dout.p, whole_lines_f32(head_dim));
    rc = st.commit(err);
    if (rc) return rc;
    rc = mha_masked_device(nullptr, (const float*)dq.p, (const float*)dk.p, (const float*)dv.p,
                           mask_len ? (const float*)dm.p : nullptr, mask_len, (float*)dout.p, batch, t_q, t_kv, heads,
                           head_dim, err);
    if (rc) return rc;
    return st.fetch(err);
} RT_NO_THROW

RT_API int rt_mha_forward_masked_f32_dev(void* stream, const float* q, const float* k, const float* v, const float* mask,
                                         size_t mask_len, float* out, size_t batch, size_t t_q, size_t t_kv,
                                         size_t heads, size_t head_dim, rt_err_detail* err) {
    clear_err(err);
    if (head_dim == 0) return fail(err, RT_ERR_ZERO_DIM, -1, 0, 0, "dim must be > 0");
    const size_t embed = heads * head_dim;
    const size_t q_expected = batch * t_q * embed, kv_expected = batch * t_kv * embed;
    const size_t one_mask = t_q * t_kv, all_masks = batch * heads * one_mask;
    if (!mask) mask_len = 0;
    if (mask_len != 0 && mask_len != one_mask && mask_len != all_masks)
        return fail(err, RT_ERR_WRONG_INPUT_LEN, RT_WHICH_MASK, one_mask, mask_len, "mask length");
    if (q_expected == 0) return RT_OK;
    if (!q || !out || (kv_expected && (!k || !v))) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    if (head_dim > 512) return fail(err, RT_ERR_UNSUPPORTED, -1, 512, head_dim, "rows kernel covers dim <= 512");
    if (heads > 65535 || batch > 65535 || t_q > 0x7fffffffull || t_kv > 0x7fffffffull || embed > 0x7fffffffull)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, 0, "shape too large for the launch grid");
    int rc = ensure_device(err);
    if (rc) return rc;
    return mha_masked_device((hipStream_t)stream, q, k, v, mask_len ? mask : nullptr, mask_len, out, batch, t_q, t_kv,
                             heads, head_dim, err);
}

// bf16 counterpart of rt_mha_forward_masked_f32_dev: steps 2-8 of MultiHeadAttention::forward's composed path
// (crates/rustorch-nn/src/attention.rs:371-399) on bf16 [B,T,H*hd] tensors with an f32 additive mask.
RT_API int rt_mha_forward_masked_bf16_dev(void* stream, const void* q, const void* k, const void* v, const float* mask,
                                          size_t mask_len, void* out, size_t batch, size_t t_q, size_t t_kv,
                                          size_t heads, size_t head_dim, rt_err_detail* err) {
    clear_err(err);
    if (head_dim == 0) return fail(err, RT_ERR_ZERO_DIM, -1, 0, 0, "dim must be > 0");
    const size_t embed = heads * head_dim;
    const size_t q_expected = batch * t_q * embed, kv_expected = batch * t_kv * embed;
    const size_t one_mask = t_q * t_kv, all_masks = batch * heads * one_mask;
    if (!mask) mask_len = 0;
    if (mask_len != 0 && mask_len != one_mask && mask_len != all_masks)
        return fail(err, RT_ERR_WRONG_INPUT_LEN, RT_WHICH_MASK, one_mask, mask_len, "mask length");
    if (q_expected == 0) return RT_OK;
    if (!q || !out || (kv_expected && (!k || !v))) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    if (head_dim > 512) return fail(err, RT_ERR_UNSUPPORTED, -1, 512, head_dim, "bf16 kernels cover head dims up to 512");
    if (heads > 65535 || batch > 65535 || t_q > 0x7fffffffull || t_kv > 0x7fffffffull || embed > 0x7fffffffull ||
        (t_q + 127) / 128 > 65535)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, 0, "shape too large for the launch grid");
    if (((uintptr_t)mask & 3) != 0) return fail(err, RT_ERR_UNSUPPORTED, -1, 4, 0, "the mask must be 4-byte aligned");
    int rc = ensure_device(err);
    if (rc) return rc;
    if (!rt::flash_tile_bf16_supported((int)head_dim) || (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15) != 0 ||
        !rt::flash_tile_bf16_addressable((long long)t_kv, (long long)(heads * head_dim)) ||
        (mask_len && !rt::flash_tile_bf16_bias_addressable((long long)t_kv))) {
        // head dims and alignments the matrix-core kernel does not cover: one workgroup per query row, any speed
        if (t_kv == 0) return rt_buf_zero(out, q_expected * 2, stream, err);
        rt::AttnRowsParams r{};
        r.q = q;
        r.k = k;
        r.v = v;
        r.out = out;
        r.batch = (int)batch;
        r.heads = r.kv_heads = (int)heads;
        r.seq_q = (int)t_q;
        r.kv_len = r.kv_stride = (int)t_kv;
        r.dim = (int)head_dim;
        r.head_map = 0;
        r.scale = 1.0f / sqrtf((float)head_dim);
        r.bias = mask_len ? mask : nullptr;
        r.bias_bh_stride = (mask_len == all_masks && all_masks != one_mask) ? (long long)one_mask : 0;
        r.use_layout = 1;
        r.lq = r.lo = rt::layout_bnhd((long long)heads, (long long)t_q, (int)head_dim);
        r.lkv = rt::layout_bnhd((long long)heads, (long long)t_kv, (int)head_dim);
        HIP_TRY(rt::launch_attn_rows_bf16((hipStream_t)stream, r), "attn_rows_bf16 launch");
        return RT_OK;
    }
    rt::FlashTileParams t{};
    t.q = (const uint16_t*)q;
    t.k = (const uint16_t*)k;
    t.v = (const uint16_t*)v;
    t.out = (uint16_t*)out;
    t.bias = mask_len ? mask : nullptr;
    t.bias_bh_stride = (mask_len == all_masks && all_masks != one_mask) ? (long long)one_mask : 0;
    t.bias_vec4 = (((uintptr_t)mask & 15) == 0 && t_kv % 4 == 0) ? 1 : 0;
    t.batch = (int)batch;
    t.heads = t.kv_heads = (int)heads;
    t.group = 1;
    t.pack = 1;
    t.n_cus = g_num_cus;
    t.seq_q = (int)t_q;
    t.seq_kv = (int)t_kv;
    t.dim = (int)head_dim;
    t.mask = rt::kMaskNone;
    t.ref_bc = 64;
    t.zero_padded_rows = 0;
    t.scale = 1.0f / sqrtf((float)head_dim);
    t.scale_log2e = t.scale * rt::kLog2eHost;
    t.lq = t.lo = rt::layout_bnhd((long long)heads, (long long)t_q, (int)head_dim);
    t.lkv = rt::layout_bnhd((long long)heads, (long long)t_kv, (int)head_dim);
    if (t_kv == 0)  // no key to weigh: the reference's products over an empty axis leave rows of zeros
        return rt_buf_zero(out, q_expected * 2, stream, err);
    HIP_TRY(rt::launch_flash_tile_bf16((hipStream_t)stream, t), "flash_tile_bf16 launch");
    return RT_OK;
}

// Causal attention with a sliding window on bf16 tensors, the mask itself never built: position i sees keys
// (i - window, i].  bnhd: [batch, seq, heads, dim] tensors (MultiHeadAttention's), else [batch, heads, seq, dim].
static int flash_window_bf16(void* stream, const rt_attention_shape* shape, uint64_t n_kv_heads, const void* q, const void* k,
                             const void* v, uint64_t window, void* out, rt_err_detail* err, bool bnhd) {
    clear_err(err);
    if (!shape) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "shape is NULL");
    if (shape->dim == 0) return fail(err, RT_ERR_ZERO_DIM, -1, 0, 0, "dim must be > 0");
    if (window == 0) return fail(err, RT_ERR_UNSUPPORTED, -1, 1, 0, "window must be >= 1 (masks.rs:51)");
    if (n_kv_heads == 0) n_kv_heads = shape->heads;
    if (shape->seq == 0 || shape->batch == 0 || shape->heads == 0) return RT_OK;
    int rc = check_flash_dims(shape, n_kv_heads, err);
    if (rc) return rc;
    if (shape->heads > 65535 || shape->batch > 65535 || (shape->seq + 127) / 128 > 65535)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, 0, "shape too large for the launch grid");
    if (!q || !k || !v || !out) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    if (!rt::flash_tile_bf16_supported((int)shape->dim))
        return fail(err, RT_ERR_UNSUPPORTED, -1, 256, shape->dim,
                    "the windowed kernel covers head dims up to 256 that are a multiple of 8 (others: the additive-mask entry)");
    if ((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15) != 0)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 16, 0, "bf16 kernels need 16-byte aligned tensors");
    if (!rt::flash_tile_bf16_addressable((long long)shape->seq, (long long)((bnhd ? n_kv_heads : 1) * shape->dim)))
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, shape->seq, "a K/V slab of one (batch, kv head) must stay below 4 GiB");
    rc = ensure_device(err);
    if (rc) return rc;
    const int dim = (int)shape->dim;
    rt::FlashTileParams t{};
    t.q = (const uint16_t*)q;
    t.k = (const uint16_t*)k;
    t.v = (const uint16_t*)v;
    t.out = (uint16_t*)out;
    t.batch = (int)shape->batch;
    t.heads = (int)shape->heads;
    t.kv_heads = (int)n_kv_heads;
    t.group = (int)(shape->heads / n_kv_heads);
    t.pack = 1;
    t.n_cus = g_num_cus;
    t.seq_q = t.seq_kv = (int)shape->seq;
    t.dim = dim;
    t.mask = rt::kMaskCausal;
    t.ref_bc = 64;
    t.scale = 1.0f / sqrtf((float)dim);
    t.scale_log2e = t.scale * rt::kLog2eHost;
    t.window = (int)(window > shape->seq ? shape->seq : window);  // a window of the whole sequence and more is the causal mask
    if (bnhd) {
        t.lq = t.lo = rt::layout_bnhd((long long)shape->heads, (long long)shape->seq, dim);
        t.lkv = rt::layout_bnhd((long long)n_kv_heads, (long long)shape->seq, dim);
    } else {
        t.lq = t.lo = rt::layout_bhnd((long long)shape->heads, (long long)shape->seq, dim);
        t.lkv = rt::layout_bhnd((long long)n_kv_heads, (long long)shape->seq, dim);
    }
    HIP_TRY(rt::launch_flash_tile_bf16((hipStream_t)stream, t), "flash_tile_bf16 (window) launch");
    return RT_OK;
}

RT_API int rt_flash_forward_window_bf16_dev(void* stream, const rt_attention_shape* shape, uint64_t n_kv_heads, const void* q,
                                            const void* k, const void* v, uint64_t window, void* out, rt_err_detail* err) {
    return flash_window_bf16(stream, shape, n_kv_heads, q, k, v, window, out, err, false);
}

RT_API int rt_flash_forward_window_bnhd_bf16_dev(void* stream, const rt_attention_shape* shape, uint64_t n_kv_heads,
                                                 const void* q, const void* k, const void* v, uint64_t window, void* out,
                                                 rt_err_detail* err) {
    return flash_window_bf16(stream, shape, n_kv_heads, q, k, v, window, out, err, true);
}

RT_API int rt_flash_forward_varlen_bf16_dev(void* stream, const rt_attention_shape* shape, uint64_t n_kv_heads,
                                            const void* q, const void* k, const void* v, const int32_t* seq_lens,
                                            int zero_padded_rows, void* out, rt_err_detail* err) {
    return flash_bf16_common(stream, shape, n_kv_heads, q, k, v, rt::kMaskVarlenCausal, nullptr, seq_lens,
                             zero_padded_rows, out, err);
}

// ---- decode, device pointers -------------------------------------------------------------------------

RT_API int rt_kv_append_bf16(void* stream, void* k_cache, void* v_cache, const void* k_in, const void* v_in,
                             int32_t pos, int32_t n_kv, int32_t head_dim, int32_t max_seq, rt_err_detail* err) {
    clear_err(err);
    if (n_kv < 0 || head_dim < 0 || max_seq < 0) return fail(err, RT_ERR_UNSUPPORTED, -1, 0, 0, "negative dimension");
    if (pos < 0 || pos >= max_seq)
        return fail(err, RT_ERR_KV_OVERFLOW, -1, (uint64_t)max_seq, (uint64_t)(int64_t)pos + 1, "position outside the cache");
    if (n_kv == 0 || head_dim == 0) return RT_OK;
    if (!k_cache || !v_cache || !k_in || !v_in) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    int rc = ensure_device(err);
    if (rc) return rc;
    HIP_TRY(rt::launch_kv_append_bf16((hipStream_t)stream, (uint16_t*)k_cache, (uint16_t*)v_cache,
                                      (const uint16_t*)k_in, (const uint16_t*)v_in, pos, n_kv, head_dim, max_seq),
            "kv_append_bf16 launch");
    return RT_OK;
}

RT_API int rt_kv_cache_append_dev(void* stream, void* k_cache, void* v_cache, const void* new_k, size_t new_k_len,
                                  const void* new_v, size_t new_v_len, size_t batch, size_t n_heads, size_t max_seq,
                                  size_t head_dim, size_t current_len, size_t seq_added, size_t elem_bytes,
                                  rt_err_detail* err) {
    clear_err(err);
    if (current_len + seq_added > max_seq)  // kv_cache.rs:84-89
        return fail(err, RT_ERR_KV_OVERFLOW, -1, (uint64_t)max_seq, (uint64_t)(current_len + seq_added), "append beyond max_seq");
    const size_t bhsd = batch * n_heads * seq_added * head_dim;
    if (new_k_len != bhsd || new_v_len != bhsd) {  // kv_cache.rs:90-97
        int rc = fail(err, RT_ERR_KV_WRONG_INPUT_LEN, -1, (uint64_t)bhsd, (uint64_t)new_k_len, "new_k / new_v length");
        if (err) err->got2 = (uint64_t)new_v_len;
        return rc;
    }
    if (elem_bytes != 2 && elem_bytes != 4) return fail(err, RT_ERR_UNSUPPORTED, -1, 0, (uint64_t)elem_bytes, "elem_bytes must be 2 or 4");
    if (batch * n_heads > 65535) return fail(err, RT_ERR_UNSUPPORTED, -1, 0, 0, "shape too large for the launch grid");
    if (bhsd == 0) return RT_OK;
    if (!k_cache || !v_cache || !new_k || !new_v) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    int rc = ensure_device(err);
    if (rc) return rc;
    HIP_TRY(rt::launch_kv_block_append((hipStream_t)stream, k_cache, v_cache, new_k, new_v, batch * n_heads, max_seq, head_dim,
                                       current_len, seq_added, elem_bytes),
            "kv_cache_append launch");
    return RT_OK;
}

RT_API int rt_qk_norm_rope_kv_append_bf16(void* stream, void* q, const void* k_in, const void* v_in, void* k_cache,
                                          void* v_cache, const int32_t* positions, int32_t pos, const float* q_gamma,
                                          const float* k_gamma, float eps, const float* cos_table,
                                          const float* sin_table, int32_t table_rows, int32_t batch, int32_t seq,
                                          int32_t n_heads, int32_t n_kv, int32_t head_dim, int32_t max_seq,
                                          rt_err_detail* err) {
    clear_err(err);
    if (batch < 0 || seq < 0 || n_heads < 0 || n_kv < 0 || head_dim < 0 || max_seq < 0 || table_rows < 0)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, 0, "negative dimension");
    if ((head_dim & 1) || head_dim > 512)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 512, (uint64_t)head_dim, "head_dim must be even and <= 512");
    if (batch > 65535 || seq > 65535 || n_heads + n_kv > 65535)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, 0, "shape too large for the launch grid");
    if (!positions) {
        // the checks of RoPE::apply_inplace_half_split (rope.rs:179-184), then of KVLayerCache::append (kv_cache.rs:84-89)
        if (pos < 0 || (int64_t)pos + seq > table_rows)
            return fail(err, RT_ERR_ROPE_POSITION_OVERFLOW, -1, (uint64_t)table_rows, (uint64_t)((int64_t)pos + seq),
                        "positions outside the RoPE tables");
        if ((int64_t)pos + seq > max_seq)
            return fail(err, RT_ERR_KV_OVERFLOW, -1, (uint64_t)max_seq, (uint64_t)((int64_t)pos + seq), "rows outside the cache");
    }
    if (batch == 0 || seq == 0 || n_heads + n_kv == 0 || head_dim == 0) return RT_OK;
    if ((n_heads > 0 && !q) || (n_kv > 0 && (!k_in || !v_in || !k_cache || !v_cache)) || !cos_table || !sin_table)
        return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    int rc = ensure_device(err);
    if (rc) return rc;
    rt::DecodePrepareParams p;
    p.q = (uint16_t*)q;
    p.k_in = (const uint16_t*)k_in;
    p.v_in = (const uint16_t*)v_in;
    p.k_cache = (uint16_t*)k_cache;
    p.v_cache = (uint16_t*)v_cache;
    p.positions = positions;
    p.q_gamma = q_gamma;
    p.k_gamma = k_gamma;
    p.cos_table = cos_table;
    p.sin_table = sin_table;
    p.eps = eps;
    p.pos = pos;
    p.batch = batch;
    p.seq = seq;
    p.n_heads = n_heads;
    p.n_kv = n_kv;
    p.head_dim = head_dim;
    p.max_seq = max_seq;
    p.table_rows = table_rows;
    HIP_TRY(rt::launch_decode_prepare((hipStream_t)stream, p), "decode_prepare launch");
    return RT_OK;
}

static int check_decode_dims(int32_t batch, int32_t n_heads, int32_t n_kv, int32_t head_dim, int32_t max_seq,
                             rt_err_detail* err) {
    if (batch < 0 || n_heads < 0 || n_kv < 0 || head_dim < 0 || max_seq < 0)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, 0, "negative dimension");
    if (n_kv == 0 || n_heads % n_kv != 0)
        return fail(err, RT_ERR_HEAD_COUNT_MISMATCH, -1, (uint64_t)n_heads, (uint64_t)n_kv,
                    "n_heads not divisible by n_kv");
    if (head_dim == 0) return fail(err, RT_ERR_ZERO_DIM, -1, 0, 0, "head_dim must be > 0");
    if (batch > 65535 || n_heads > 65535) return fail(err, RT_ERR_UNSUPPORTED, -1, 0, 0, "shape too large for the launch grid");
    return RT_OK;
}

// Scratch of a single-sequence decode (p.ws, p.n_waves, p.compact).
static int online_scratch(hipStream_t stream, rt::DecodeSplitParams& p, rt_err_detail* err) {
    size_t slot_bytes = 0;
    int rc = stream_slot_scratch(stream, &p.ws, &slot_bytes, err);
    if (rc) return rc;
    if (p.ws) {
        // compact numbering: (waves + kv heads) * group partials of dim + 2 floats
        const size_t per_wave = (size_t)(p.heads / p.kv_heads) * ((size_t)p.dim + 2) * sizeof(float);
        const long long fit = (long long)(slot_bytes / per_wave) - p.kv_heads;
        if (fit >= std::min<long long>(p.n_waves, 256)) {
            p.n_waves = (int)std::min<long long>(p.n_waves, fit);
            p.compact = 1;
            return RT_OK;
        }
    }
    return stream_workspace(stream, rt::decode_split_workspace_bytes(1, p.heads, p.dim, p.max_seq), &p.ws, err);
}

RT_API int rt_gqa_decode_online_bf16(void* stream, const void* q, const void* k_cache, const void* v_cache,
                                     void* out, int32_t n_heads, int32_t n_kv, int32_t kv_len, int32_t head_dim,
                                     int32_t max_seq, rt_err_detail* err) try {
    clear_err(err);
    int rc = check_decode_dims(1, n_heads, n_kv, head_dim, max_seq, err);
    if (rc) return rc;
    if (kv_len < 0 || kv_len > max_seq)
        return fail(err, RT_ERR_KV_OVERFLOW, -1, (uint64_t)max_seq, (uint64_t)(int64_t)kv_len, "kv_len outside the cache");
    if (n_heads == 0) return RT_OK;
    if (head_dim > 512) return fail(err, RT_ERR_UNSUPPORTED, -1, 512, (uint64_t)head_dim, "decode rows kernel covers dim <= 512");
    if (!q || !out || (kv_len > 0 && (!k_cache || !v_cache))) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    rc = ensure_device(err);
    if (rc) return rc;
    // the split-K kernels move q, K and V 16 bytes at a time; tensors that are not 16-byte aligned take the
    // element-wise kernel below
    const bool aligned = ((((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15) == 0);
    if (aligned && rt::decode_split_supported(n_heads, n_kv, head_dim)) {
        // the split-K kernels of the batched entry, on a batch of one
        rt::DecodeSplitParams sp{};
        sp.span_min = rt::decode_split_span_min(1);
        // no more one-wave workgroups than there are spans of the minimum length (short contexts)
        const long long steps = (long long)n_kv * ((kv_len + 31) / 32);
        const long long spans = (steps + sp.span_min - 1) / sp.span_min;
        sp.n_waves = (int)std::min<long long>(g_decode_waves, std::max<long long>(spans, 1));
        sp.q = (const uint16_t*)q;
        sp.k_cache = (const uint16_t*)k_cache;
        sp.v_cache = (const uint16_t*)v_cache;
        sp.out = (uint16_t*)out;
        sp.kv_lens = nullptr;
        sp.kv_len = kv_len;
        sp.batch = 1;
        sp.heads = n_heads;
        sp.kv_heads = n_kv;
        sp.dim = head_dim;
        sp.max_seq = max_seq;
        sp.n_part = rt::decode_split_parts(1, max_seq);
        sp.scale_log2e = (1.0f / sqrtf((float)head_dim)) * rt::kLog2eHost;
        rc = plan_decode((hipStream_t)stream, sp, kv_len, err);
        if (rc) return rc;
        // The reference's signature has no workspace argument: the partials go to this stream's slot of the library's fixed
        // scratch block (nothing is allocated, so the call can be captured into a graph), in the compact slot numbering;
        // only when no slot is free, or the slot cannot hold a useful number of partials, to a buffer the library
        // allocates per stream.  Where neither may be used: one split, which leaves no partials, if the output is aligned for it.
        ScratchTurn turn;
        if (sp.n_splits != 1) {
            bool scratch = false;
            rc = turn.enter((hipStream_t)stream, &scratch, err);
            if (rc) return rc;
            if (scratch) {
                rc = online_scratch((hipStream_t)stream, sp, err);
                if (rc) return rc;
            } else if (((uintptr_t)out & 7) == 0) {
                sp.n_splits = 1;
            }
        }
        if (sp.ws || sp.n_splits == 1) {
            HIP_TRY(rt::launch_decode_split((hipStream_t)stream, sp), "decode_split launch");
            return turn.leave((hipStream_t)stream, err);
        }
    }
    rt::AttnRowsParams p{};
    p.q = q;
    p.k = k_cache;
    p.v = v_cache;
    p.out = out;
    p.kv_lens = nullptr;
    p.batch = 1;
    p.heads = n_heads;
    p.kv_heads = n_kv;
    p.seq_q = 1;
    p.kv_len = kv_len;
    p.kv_stride = max_seq;
    p.dim = head_dim;
    p.head_map = 1;
    p.scale = 1.0f / sqrtf((float)head_dim);
    HIP_TRY(rt::launch_attn_rows_bf16((hipStream_t)stream, p), "attn_rows_bf16 launch");
    return RT_OK;
} RT_NO_THROW

RT_API int rt_gqa_decode_naive_bf16(void* stream, const void* q, const void* k_cache, const void* v_cache, void* out,
                                    int32_t n_heads, int32_t n_kv, int32_t kv_len, int32_t head_dim, int32_t max_seq,
                                    rt_err_detail* err) {
    return rt_gqa_decode_online_bf16(stream, q, k_cache, v_cache, out, n_heads, n_kv, kv_len, head_dim, max_seq, err);
}

namespace {
// Into how many spans the keys of a chunk's units are cut: the cheapest of a workgroup's tile steps (0.75 us at head dim 64,
// 1.1 at 128, with a CU to itself, half as much again for every workgroup that shares it; above head dim 64, where no third one
// covers its set-up, each costs 0.8 us besides) plus, when there are spans, the merge launch (3 us) and the partials' way to memory
// and back (3 TB/s).  Over 36 shapes (2 to 341 positions, 130 to 8192 keys, head dims 64 to 256) its choice is within 2 % of
// the best count measured.  One sequence, 32 heads over 8 of 128, 8192 keys: 16 positions 119 -> 14.9 us (32 spans), 100
// positions 28.5 (8).  Short walks are cut to single tiles: 16 heads of 64, 2 positions over 900 keys, us by spans 1 16.3, 5 10.1,
// 8 9.3, 15 7.9; 8 x 16 heads of 64, 4 over 800, 1 14.6, 2 14.2, 4 12.6; 32 / 8 of 128, 4 over 200, 1 9.6, 4 8.6; but, for their
// partials, 16 over 1000, 8 10.5, 16 10.9.
// Units that fill the chip by themselves are not cut.
// Above head dim 128 all of it is the times of tiles through registers, 32 keys each.  Where a span takes tiles of 64 straight to LDS instead
// (flash_tile_bf16_direct) the counts are as good: of those measured over 23 shapes the choice is within 5 % of the best, but for two
// (12 and 14 %).  A last span that 64 keys leave empty stays: with one span less, sequences, positions, heads, head
// dim, keys, spans: 2 54 16/2 160 6507 16 28.0, 15 25.0; but 1 64 28/4 160 4234 15 23.0, 14 25.2; 1 161 8/2 256 5973 17 26.0, 16 29.4; 3 39 8/2 160 7262 21
// 23.4, 20 22.7, 19 23.2.
long long chunk_splits(long long slabs, long long rows, int head_dim, long long keys) {
    const long long key_tile = rt::flash_tile_bf16_key_tile(head_dim, false), tiles = (keys + key_tile - 1) / key_tile;
    const long long units = slabs * ((rows + 127) / 128);
    if (units >= g_num_cus || tiles < 4) return 1;
    const long long occ = rt::flash_tile_bf16_workgroups(head_dim);
    const float step_us = 0.4f + 0.7f * (float)key_tile * (float)head_dim / (64.0f * 128.0f);
    const float partial_us = (float)(slabs * rows) * (float)(head_dim + 2) * (2 * sizeof(float)) / 3.0e6f;
    long long best = 1;
    float best_us = 0.0f;
    for (long long n = 1; n <= std::min<long long>(tiles, 64) && (n - 1) * units < occ * g_num_cus; n++) {
        const long long per_cu = (units * n + g_num_cus - 1) / g_num_cus, rounds = per_cu / occ, rest = per_cu % occ;
        const float load = 0.5f * (float)(rounds * (occ + 1) + (rest ? rest + 1 : 0));
        const float us = (float)((tiles + n - 1) / n) * step_us * load + (head_dim > 64 ? 1.6f * (load - 1.0f) : 0.0f) +
                         (n > 1 ? 3.0f + (float)n * partial_us : 0.0f);
        if (n == 1 || us < best_us) {
            best = n;
            best_us = us;
        }
    }
    return best;
}
}  // namespace

// Several new positions per sequence against the cache, causally masked: the bf16 form of gqa_decode_batched_f32
// (crates/rustorch-metal/src/kernels.rs:14432-14516), batched over sequences with their own context lengths.
RT_API int rt_gqa_decode_chunk_bf16(void* stream, const void* q, const void* k_cache, const void* v_cache, void* out,
                                    const int32_t* kv_lens, int32_t kv_len, int32_t batch, int32_t seq_new,
                                    int32_t n_heads, int32_t n_kv, int32_t head_dim, int32_t max_seq,
                                    rt_err_detail* err) try {
    clear_err(err);
    int rc = check_decode_dims(batch, n_heads, n_kv, head_dim, max_seq, err);
    if (rc) return rc;
    if (seq_new < 0) return fail(err, RT_ERR_UNSUPPORTED, -1, 0, 0, "negative dimension");
    if (!kv_lens && (kv_len < seq_new || kv_len > max_seq))
        return fail(err, RT_ERR_KV_OVERFLOW, -1, (uint64_t)max_seq, (uint64_t)(int64_t)kv_len,
                    "kv_len must cover the new positions and fit the cache");
    if (batch == 0 || n_heads == 0 || seq_new == 0) return RT_OK;
    if (!q || !out || !k_cache || !v_cache) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    if (!rt::flash_tile_bf16_supported(head_dim))
        return fail(err, RT_ERR_UNSUPPORTED, -1, 256, (uint64_t)head_dim,
                    "bf16 kernels cover head dims up to 256 that are a multiple of 8");
    if ((((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)out) & 15) != 0)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 16, 0, "bf16 kernels need 16-byte aligned tensors");
    if (!rt::flash_tile_bf16_addressable((long long)max_seq, (long long)head_dim))
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, (uint64_t)max_seq, "a cache slab of one (sequence, kv head) must stay below 4 GiB");
    const int group = n_heads / n_kv;
    if (((int64_t)seq_new * group + 127) / 128 > 65535 || batch > 65535 || n_kv > 65535)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, 0, "shape too large for the launch grid");
    rc = ensure_device(err);
    if (rc) return rc;
    rt::FlashTileParams t{};
    t.q = (const uint16_t*)q;
    t.k = (const uint16_t*)k_cache;
    t.v = (const uint16_t*)v_cache;
    t.out = (uint16_t*)out;
    t.kv_lens = kv_lens;
    t.batch = batch;
    t.heads = n_heads;
    t.kv_heads = n_kv;
    t.group = group;
    t.pack = group;  // rows of a tile run over (position, head of the group): one pass over a kv head's keys serves them all
    t.decode_rows = 1;  // (also with one head per group: a position without keys is a row of zeros)
    t.seq_q = seq_new;
    t.seq_kv = kv_lens ? max_seq : kv_len;
    t.dim = head_dim;
    t.mask = rt::kMaskCausal;  // position s sees keys [0, kv_len - seq_new + s]
    t.ref_bc = 64;
    t.zero_padded_rows = 0;
    t.scale = 1.0f / sqrtf((float)head_dim);
    t.scale_log2e = t.scale * rt::kLog2eHost;
    t.lq = t.lo = rt::layout_bnhd((long long)n_heads, (long long)seq_new, head_dim);
    t.lkv = rt::layout_bhnd((long long)n_kv, (long long)max_seq, head_dim);
    // Few (sequence, kv head, query tile) units and a long cache -- the reference's own call shape, one sequence: cut the
    // keys into spans (chunk_splits).  The partials go to this stream's slot of the library's fixed scratch block where
    // it holds them, else to the buffer the library keeps per stream; under capture, where that one cannot be allocated,
    // to as many spans as the slot holds.
    const long long rows = (long long)seq_new * group;
    long long n_splits = chunk_splits((long long)batch * n_kv, rows, head_dim, t.seq_kv);
    float* ws = nullptr;
    const size_t part_rows = (size_t)batch * n_kv * (size_t)((rows + 31) / 32 * 32);
    const size_t per_split = part_rows * ((size_t)head_dim + 2) * sizeof(float);
    ScratchTurn turn;
    if (n_splits > 1) {
        bool scratch = false;
        rc = turn.enter((hipStream_t)stream, &scratch, err);
        if (rc) return rc;
        if (!scratch) n_splits = 1;
    }
    if (n_splits > 1) {
        size_t slot_bytes = 0;
        rc = stream_slot_scratch((hipStream_t)stream, &ws, &slot_bytes, err);
        if (rc) return rc;
        if (!ws || slot_bytes < per_split * (size_t)n_splits) {
            bool captured = false;
            if (ws) rc = is_capturing((hipStream_t)stream, &captured, err);
            if (rc) return rc;
            float* kept = nullptr;
            if (!captured) {
                rc = stream_workspace((hipStream_t)stream, per_split * (size_t)n_splits, &kept, err);
                if (rc && !ws) return rc;
                clear_err(err);
            }
            if (kept) ws = kept;
            else n_splits = (long long)(slot_bytes / per_split);  // (below two: the call runs without partials)
        }
    }
    if (n_splits > 1) {
        t.n_splits = (int)n_splits;
        t.part_o = ws;
        t.part_ml = ws + part_rows * (size_t)n_splits * (size_t)head_dim;
    }
    HIP_TRY(rt::launch_flash_tile_bf16((hipStream_t)stream, t), "flash_tile_bf16 launch");
    return turn.leave((hipStream_t)stream, err);
} RT_NO_THROW

RT_API size_t rt_gqa_decode_workspace_bytes(int32_t batch, int32_t n_heads, int32_t n_kv, int32_t head_dim,
                                            int32_t max_seq) {
    if (batch <= 0 || n_heads <= 0 || n_kv <= 0 || head_dim <= 0 || max_seq < 0) return 0;
    if (!rt::decode_split_supported(n_heads, n_kv, head_dim)) return 0;
    return rt::decode_split_workspace_bytes(batch, n_heads, head_dim, max_seq);
}

RT_API int rt_gqa_decode_batched_bf16(void* stream, const void* q, const void* k_cache, const void* v_cache,
                                      void* out, const int32_t* kv_lens, int32_t batch, int32_t n_heads,
                                      int32_t n_kv, int32_t head_dim, int32_t max_seq, void* workspace,
                                      size_t workspace_bytes, rt_err_detail* err) {
    clear_err(err);
    int rc = check_decode_dims(batch, n_heads, n_kv, head_dim, max_seq, err);
    if (rc) return rc;
    if (batch == 0 || n_heads == 0) return RT_OK;
    if (!q || !out || !kv_lens || (max_seq > 0 && (!k_cache || !v_cache)))
        return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    rc = ensure_device(err);
    if (rc) return rc;
    // the split-K kernels move q, K, V and the partials 16 bytes at a time; tensors that are not 16-byte aligned
    // take the element-wise kernel below, which needs no workspace
    const bool aligned = ((((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15) == 0);
    if (aligned && rt::decode_split_supported(n_heads, n_kv, head_dim)) {
        size_t need = rt::decode_split_workspace_bytes(batch, n_heads, head_dim, max_seq);
        if (!workspace || workspace_bytes < need)
            return fail(err, RT_ERR_WORKSPACE_TOO_SMALL, -1, need, workspace ? workspace_bytes : 0, "workspace too small");
        if ((uintptr_t)workspace & 15)
            return fail(err, RT_ERR_WORKSPACE_TOO_SMALL, -1, 16, (uint64_t)((uintptr_t)workspace & 15),
                        "workspace must be 16-byte aligned");
        rt::DecodeSplitParams p{};
        p.q = (const uint16_t*)q;
        p.k_cache = (const uint16_t*)k_cache;
        p.v_cache = (const uint16_t*)v_cache;
        p.out = (uint16_t*)out;
        p.kv_lens = kv_lens;
        p.ws = (float*)workspace;
        p.batch = batch;
        p.heads = n_heads;
        p.kv_heads = n_kv;
        p.dim = head_dim;
        p.max_seq = max_seq;
        p.n_part = rt::decode_split_parts(batch, max_seq);
        p.span_min = rt::decode_split_span_min(batch);
        p.n_waves = g_decode_waves;
        p.scale_log2e = (1.0f / sqrtf((float)head_dim)) * rt::kLog2eHost;
        rc = plan_decode((hipStream_t)stream, p, max_seq, err);
        if (rc) return rc;
        HIP_TRY(rt::launch_decode_split((hipStream_t)stream, p), "decode_split launch");
        return RT_OK;
    }
    // shapes outside the split-K kernel: one workgroup per (sequence, head), no workspace
    if (head_dim > 512) return fail(err, RT_ERR_UNSUPPORTED, -1, 512, (uint64_t)head_dim, "decode rows kernel covers dim <= 512");
    rt::AttnRowsParams p{};
    p.q = q;
    p.k = k_cache;
    p.v = v_cache;
    p.out = out;
    p.kv_lens = kv_lens;
    p.batch = batch;
    p.heads = n_heads;
    p.kv_heads = n_kv;
    p.seq_q = 1;
    p.kv_len = 0;
    p.kv_stride = max_seq;
    p.dim = head_dim;
    p.head_map = 1;
    p.scale = 1.0f / sqrtf((float)head_dim);
    HIP_TRY(rt::launch_attn_rows_bf16((hipStream_t)stream, p), "attn_rows_bf16 launch");
    return RT_OK;
}

// The batched decode for callers that cannot allocate (under HIP graph capture, in serving loops or harnesses that
// forbid hipMalloc): the partials go to the library's fixed scratch block in device memory instead of a workspace
// argument.  Calls nothing that allocates or frees.
RT_API int rt_gqa_decode_batched_bf16_noalloc(void* stream, const void* q, const void* k_cache, const void* v_cache,
                                              void* out, const int32_t* kv_lens, int32_t batch, int32_t n_heads,
                                              int32_t n_kv, int32_t head_dim, int32_t max_seq, rt_err_detail* err) {
    clear_err(err);
    int rc = check_decode_dims(batch, n_heads, n_kv, head_dim, max_seq, err);
    if (rc) return rc;
    if (batch == 0 || n_heads == 0) return RT_OK;
    if (!q || !out || !kv_lens || (max_seq > 0 && (!k_cache || !v_cache)))
        return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    rc = ensure_device(err);
    if (rc) return rc;
    if (!rt::decode_split_supported(n_heads, n_kv, head_dim))
        return fail(err, RT_ERR_UNSUPPORTED, -1, 0, (uint64_t)head_dim,
                    "the no-allocation decode covers head_dim 64, 128, 256 with at most 16 query heads per kv head");
    if ((((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15) != 0)
        return fail(err, RT_ERR_UNSUPPORTED, -1, 16, 0, "the no-allocation decode needs 16-byte aligned q and caches");
    float* scratch = nullptr;
    size_t scratch_bytes = 0;
    HIP_TRY(rt::decode_static_scratch(&scratch, &scratch_bytes), "hipGetSymbolAddress(static scratch)");
    const size_t need = rt::decode_split_compact_bytes(batch, n_heads, n_kv, head_dim, g_decode_waves);
    if (need > scratch_bytes)
        return fail(err, RT_ERR_WORKSPACE_TOO_SMALL, -1, (uint64_t)need, (uint64_t)scratch_bytes,
                    "batch too large for the library's fixed scratch block; use rt_gqa_decode_batched_bf16 with a workspace");
    rt::DecodeSplitParams p{};
    p.q = (const uint16_t*)q;
    p.k_cache = (const uint16_t*)k_cache;
    p.v_cache = (const uint16_t*)v_cache;
    p.out = (uint16_t*)out;
    p.kv_lens = kv_lens;
    p.ws = scratch;
    p.batch = batch;
    p.heads = n_heads;
    p.kv_heads = n_kv;
    p.dim = head_dim;
    p.max_seq = max_seq;
    p.n_part = rt::decode_split_parts(batch, max_seq);
    p.span_min = rt::decode_split_span_min(batch);
    p.n_waves = g_decode_waves;
    p.scale_log2e = (1.0f / sqrtf((float)head_dim)) * rt::kLog2eHost;
    p.compact = 1;
    rc = plan_decode((hipStream_t)stream, p, max_seq, err);
    if (rc) return rc;
    HIP_TRY(rt::launch_decode_split((hipStream_t)stream, p), "decode_split launch");
    return RT_OK;
}

// ---- device buffers ------------------------------------------------------------------------------------

RT_API void* rt_buf_alloc(size_t bytes, rt_err_detail* err) {
    clear_err(err);
    if (ensure_device(err) != RT_OK) return nullptr;
    void* p = nullptr;
    hipError_t e = hipMalloc(&p, bytes ? bytes : 1);
    if (e != hipSuccess) {
        fail_hip(err, e, "hipMalloc");
        return nullptr;
    }
    return p;
}

RT_API int rt_buf_free(void* ptr, rt_err_detail* err) {
    clear_err(err);
    if (!ptr) return RT_OK;
    // a buffer may go at any time -- a garbage collector's -- and so while some stream of the process is being captured,
    // where a free would end the capture with an error unless this thread says that it knows what it does
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    HIP_TRY(hipThreadExchangeStreamCaptureMode(&mode), "hipThreadExchangeStreamCaptureMode");
    const hipError_t freed = hipFree(ptr);
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    HIP_TRY(freed, "hipFree");
    return RT_OK;
}

namespace {
__global__ __launch_bounds__(256) void zero_fill_kernel(uint32_t* p, size_t n_words) {
    const size_t n4 = n_words / 4;
    uint4* p4 = (uint4*)p;
    const size_t stride = (size_t)gridDim.x * blockDim.x, t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (((uintptr_t)p & 15) == 0) {
        for (size_t i = t; i < n4; i += stride) p4[i] = make_uint4(0u, 0u, 0u, 0u);
        for (size_t i = 4 * n4 + t; i < n_words; i += stride) p[i] = 0u;
    } else {
        for (size_t i = t; i < n_words; i += stride) p[i] = 0u;
    }
}
}  // namespace

RT_API int rt_buf_zero(void* ptr, size_t bytes, void* stream, rt_err_detail* err) {
    clear_err(err);
    if (bytes == 0) return RT_OK;
    if (!ptr) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    if ((bytes & 3) || ((uintptr_t)ptr & 3)) return fail(err, RT_ERR_UNSUPPORTED, -1, 0, (uint64_t)bytes, "zero fill works on 4-byte words");
    int rc = ensure_device(err);
    if (rc) return rc;
    const size_t n_words = bytes / 4;
    const unsigned blocks = (unsigned)std::min<size_t>((n_words / 4 + 255) / 256 + 1, 4096);
    hipLaunchKernelGGL(zero_fill_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream, (uint32_t*)ptr, n_words);
    HIP_TRY(hipGetLastError(), "zero_fill launch");
    return RT_OK;
}

namespace {
__global__ __launch_bounds__(256) void i32_add_kernel(int32_t* p, size_t n, int32_t delta) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] += delta;
}
}  // namespace

RT_API int rt_i32_add_dev(void* stream, int32_t* ptr, size_t n, int32_t delta, rt_err_detail* err) {
    clear_err(err);
    if (n == 0) return RT_OK;
    if (!ptr) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    if (((uintptr_t)ptr & 3) || n > ((size_t)1 << 30)) return fail(err, RT_ERR_UNSUPPORTED, -1, 0, (uint64_t)n, "int32 add works on up to 2^30 aligned values");
    int rc = ensure_device(err);
    if (rc) return rc;
    hipLaunchKernelGGL(i32_add_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, ptr, n, delta);
    HIP_TRY(hipGetLastError(), "i32_add launch");
    return RT_OK;
}

RT_API int rt_memcpy_h2d(void* dst, const void* src, size_t bytes, void* stream, rt_err_detail* err) {
    clear_err(err);
    if (bytes == 0) return RT_OK;
    if (!dst || !src) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, (hipStream_t)stream), "hipMemcpyAsync h2d");
    return RT_OK;
}

RT_API int rt_memcpy_d2h(void* dst, const void* src, size_t bytes, void* stream, rt_err_detail* err) {
    clear_err(err);
    if (bytes == 0) return RT_OK;
    if (!dst || !src) return fail(err, RT_ERR_NULL_POINTER, -1, 0, 0, "NULL buffer");
    HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, (hipStream_t)stream), "hipMemcpyAsync d2h");
    return RT_OK;
}

RT_API int rt_stream_synchronize(void* stream, rt_err_detail* err) {
    clear_err(err);
    HIP_TRY(hipStreamSynchronize((hipStream_t)stream), "hipStreamSynchronize");
    return RT_OK;
}

RT_API void* rt_stream_create(rt_err_detail* err) {
    clear_err(err);
    if (ensure_device(err) != RT_OK) return nullptr;
    hipStream_t s = nullptr;
    hipError_t e = hipStreamCreate(&s);
    if (e != hipSuccess) {
        fail_hip(err, e, "hipStreamCreate");
        return nullptr;
    }
    return (void*)s;
}

RT_API int rt_stream_destroy(void* stream, rt_err_detail* err) {
    clear_err(err);
    if (!stream) return RT_OK;
    {
        // the library's scratch for this stream goes with it
        std::lock_guard<std::mutex> lock(g_ws_mutex);
        int dev = 0;
        if (hipGetDevice(&dev) == hipSuccess) {
            auto it = g_ws.find({dev, (hipStream_t)stream});
            if (it != g_ws.end()) {
                (void)hipStreamSynchronize((hipStream_t)stream);
                release_stream_ws(it->second);
                g_ws.erase(it);
            }
            release_stream_slot(dev, (hipStream_t)stream);
        }
    }
    HIP_TRY(hipStreamDestroy((hipStream_t)stream), "hipStreamDestroy");
    return RT_OK;
}

RT_API int rt_shutdown(rt_err_detail* err) {
    clear_err(err);
    // what the library keeps between calls: the per-stream scratch of rt_gqa_decode_online_bf16 and the staging memory
    // of the host-slice entries.  The caller makes sure no call is in flight.
    {
        std::lock_guard<std::mutex> lock(g_ws_mutex);
        for (auto& kv : g_ws) {
            if (kv.second.ptr) (void)hipStreamSynchronize(kv.first.second);
            release_stream_ws(kv.second);
        }
        g_ws.clear();
        g_slots.clear();
    }
    ScratchTurn::release();
    {
        std::lock_guard<std::mutex> lock(g_stage.mutex);
        crew().stop();
        g_stage.release();
    }
    (void)hipGetLastError();
    return RT_OK;
}
