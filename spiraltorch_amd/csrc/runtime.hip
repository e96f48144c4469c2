// Runtime half of the C ABI: init/probe, error text, device buffers, streams and events.
// Mirrors crates/st-backend-hip/src/lib.rs:148-207 (init once, shared by all threads) and the RAII
// wrappers of crates/st-backend-hip/src/real.rs:190-220,649-697, flattened to C handles.
#include <chrono>
#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "common.h"
#include "kernels.h"

namespace sthip {

namespace {
thread_local std::string g_last_error;

struct Runtime {
    std::mutex mutex;
    bool ready = false;
    int status = ST_HIP_ERR_NOT_ENABLED;
    std::string error;
    std::vector<hipDeviceProp_t> devices;
};

Runtime &runtime()
{
    static Runtime instance;
    return instance;
}
}  // namespace

int fail(int code, const char *fmt, ...)
{
    char buffer[512];
    va_list args;
    va_start(args, fmt);
    vsnprintf(buffer, sizeof buffer, fmt, args);
    va_end(args);
    g_last_error = buffer;
    return code;
}

int hip_fail(hipError_t rc, const char *ctx)
{
    (void)hipGetLastError();  // clear the sticky flag so the next call starts clean
    return fail(ST_HIP_ERR_RUNTIME, "%s: %s (%d) - %s", ctx, hipGetErrorName(rc), static_cast<int>(rc),
                hipGetErrorString(rc));
}

void clear_error() { g_last_error.clear(); }

int ensure_init()
{
    Runtime &rt = runtime();
    std::lock_guard<std::mutex> lock(rt.mutex);
    if (rt.ready) return ST_HIP_OK;
    int count = 0;
    hipError_t rc = hipGetDeviceCount(&count);
    if (rc != hipSuccess || count <= 0) {
        (void)hipGetLastError();
        return fail(ST_HIP_ERR_NOT_ENABLED, "HIP not enabled (no usable HIP device: %s)",
                    rc == hipSuccess ? "device count is 0" : hipGetErrorString(rc));
    }
    std::vector<hipDeviceProp_t> devices(static_cast<size_t>(count));
    for (int i = 0; i < count; ++i) {
        rc = hipGetDeviceProperties(&devices[static_cast<size_t>(i)], i);
        if (rc != hipSuccess) return hip_fail(rc, "hipGetDeviceProperties");
    }
    if (std::strncmp(devices[0].gcnArchName, "gfx950", 6) != 0) {
        return fail(ST_HIP_ERR_NOT_ENABLED,
                    "HIP not enabled (device 0 is %s; this library carries gfx950 code only)",
                    devices[0].gcnArchName);
    }
    // Set-up of the allocation-free entry point: the device address of its static scratch array on the current
    // GPU (other GPUs resolve theirs on their first call with that device current).
    void *scratch_address = nullptr;
    rc = noalloc_scratch(&scratch_address);
    if (rc != hipSuccess) return hip_fail(rc, "hipGetSymbolAddress(scratch)");
    rt.devices.swap(devices);
    rt.ready = true;
    return ST_HIP_OK;
}

namespace {
std::atomic<unsigned long long> g_transfers[4];  // h2d copies, h2d bytes, d2h copies, d2h bytes
}  // namespace

void count_transfer(bool to_device, size_t bytes)
{
    g_transfers[to_device ? 0 : 2].fetch_add(1, std::memory_order_relaxed);
    g_transfers[to_device ? 1 : 3].fetch_add(bytes, std::memory_order_relaxed);
}

namespace {
// Allocating and freeing are no part of a graph, and allowed while some stream of the process is being captured only where the thread
// says that it means it.
class RelaxedCapture {
  public:
    RelaxedCapture() { exchanged_ = hipThreadExchangeStreamCaptureMode(&mode_) == hipSuccess; }
    ~RelaxedCapture()
    {
        if (exchanged_) (void)hipThreadExchangeStreamCaptureMode(&mode_);
    }
    RelaxedCapture(const RelaxedCapture &) = delete;
    RelaxedCapture &operator=(const RelaxedCapture &) = delete;

  private:
    hipStreamCaptureMode mode_ = hipStreamCaptureModeRelaxed;
    bool exchanged_ = false;
};

// Never destroyed: threads may hand buffers back while the process is shutting down.
constexpr size_t kPinnedSmallest = 64u << 10;
struct PinnedPool {
    std::mutex mutex;
    PinnedBuffer idle[kPinnedMost / kPinnedSmallest];  // as many as there can be
    size_t idle_count = 0;
    size_t held = 0;  // bytes, in use or idle
    uint64_t allocations = 0;
    struct Reading {
        PinnedBuffer buffer;
        const unsigned *words;
        size_t count;
    };
    std::vector<Reading> reading;

    void collect()  // what has been read since
    {
        for (size_t i = reading.size(); i-- > 0;) {
            size_t seen = 0;
            while (seen < reading[i].count && __atomic_load_n(&reading[i].words[seen], __ATOMIC_ACQUIRE) != 0) ++seen;
            if (seen < reading[i].count) continue;
            idle[idle_count++] = reading[i].buffer;
            reading[i] = reading.back();
            reading.pop_back();
        }
    }
    void take(size_t i, PinnedBuffer *out)
    {
        *out = idle[i];
        idle[i] = idle[--idle_count];
    }
};
PinnedPool &pinned_pool()
{
    static PinnedPool *pool = new PinnedPool;
    return *pool;
}
void pinned_free(const PinnedBuffer &buffer)
{
    const RelaxedCapture relaxed;
    if (hipHostFree(buffer.ptr) != hipSuccess) (void)hipGetLastError();
}
}  // namespace

HostMemory host_memory(const void *host)
{
    hipPointerAttribute_t attributes;
    if (hipPointerGetAttributes(&attributes, host) != hipSuccess) {
        (void)hipGetLastError();
        return HostMemory::kOrdinary;
    }
    if (attributes.type == hipMemoryTypeHost) return HostMemory::kPinned;
    return attributes.type == hipMemoryTypeManaged || attributes.type == hipMemoryTypeDevice ? HostMemory::kRuntime : HostMemory::kOrdinary;
}

// The smallest idle buffer that fits and is not far too large; a new one where the pool may grow; any that fits; a new one in the
// place of smaller ones.  Nothing is freed only because a call has ended: calls that need all there is would pin their memory
// anew each time.
bool pinned_acquire(size_t bytes, PinnedBuffer *out)
{
    if (bytes > kPinnedMost) return false;
    size_t capacity = kPinnedSmallest;
    while (capacity < bytes) capacity *= 2;
    PinnedPool &pool = pinned_pool();
    for (;;) {
        PinnedBuffer doomed;
        {
            std::lock_guard<std::mutex> lock(pool.mutex);
            pool.collect();
            size_t best = pool.idle_count, smallest = pool.idle_count;
            for (size_t i = 0; i < pool.idle_count; ++i) {
                const size_t has = pool.idle[i].capacity;
                if (has >= bytes && (best == pool.idle_count || has < pool.idle[best].capacity)) best = i;
                if (smallest == pool.idle_count || has < pool.idle[smallest].capacity) smallest = i;
            }
            const bool room = pool.held + capacity <= kPinnedMost;
            if (best < pool.idle_count && (pool.idle[best].capacity <= 4 * capacity || !room)) {
                pool.take(best, out);
                return true;
            }
            if (room) {
                pool.held += capacity;
                ++pool.allocations;
                break;
            }
            if (smallest == pool.idle_count) return false;
            pool.take(smallest, &doomed);
            pool.held -= doomed.capacity;
        }
        pinned_free(doomed);
    }
    void *ptr = nullptr;
    const RelaxedCapture relaxed;
    if (hipHostMalloc(&ptr, capacity + capacity / kCopyPiece * sizeof(unsigned), hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess) {
        (void)hipGetLastError();
        std::lock_guard<std::mutex> lock(pool.mutex);
        pool.held -= capacity;
        return false;
    }
    *out = PinnedBuffer{ptr, capacity};
    return true;
}

void pinned_release(const PinnedBuffer &buffer)
{
    if (buffer.ptr == nullptr) return;
    PinnedPool &pool = pinned_pool();
    std::lock_guard<std::mutex> lock(pool.mutex);
    pool.idle[pool.idle_count++] = buffer;
}

void pinned_release_when_read(const PinnedBuffer &buffer, const unsigned *words, size_t count)
{
    PinnedPool &pool = pinned_pool();
    std::lock_guard<std::mutex> lock(pool.mutex);
    pool.reading.push_back(PinnedPool::Reading{buffer, words, count});
}

void pinned_release_idle()
{
    PinnedPool &pool = pinned_pool();
    for (;;) {
        PinnedBuffer doomed;
        {
            std::lock_guard<std::mutex> lock(pool.mutex);
            pool.collect();
            if (pool.idle_count == 0) return;
            pool.take(pool.idle_count - 1, &doomed);
            pool.held -= doomed.capacity;
        }
        pinned_free(doomed);
    }
}

namespace {
// Device memory of tensors that are used on the default stream alone: what one frees the next may take at once, for their work is
// ordered, whatever threads they belong to.  hipFree waits for the whole device instead, 6.5 µs with nothing to wait for, and waiting for the
// stream costs about two for every launch since the last wait: a call of a classifier on 64 rows, five tensors, takes 152 µs with hipFree, a
// waiting upload and a waiting read, 149 with either of the three in their way, 116 with none (the read: st_hip_memcpy_d2h).  Blocks of
// powers of two, kept for the device they are on, kTensorMost bytes at the most: the longest idle ones make room for the next, so that
// sizes a program no longer uses do not keep out those it does.  Larger ones go back to the runtime.
constexpr size_t kTensorSmallest = 4u << 10, kTensorLargest = 8u << 20, kTensorMost = 64u << 20;
struct TensorBlock {
    void *ptr;
    size_t capacity;
    size_t bytes;  // that were asked for
    int device;
    uint64_t idle_since;  // 0: in use
};
struct TensorPool {
    std::mutex mutex;
    std::map<const char *, TensorBlock> blocks;  // in use or idle; a block may be freed by a thread whose device is another
    std::deque<TensorBlock *> idle[__builtin_ctzll(kTensorLargest / kTensorSmallest) + 1];  // by size, the longest idle first
    size_t held = 0;
    uint64_t frees = 0;
    // The tensor whose memory `ptr` lies in.
    const TensorBlock *find(const void *ptr) const
    {
        const char *const at = static_cast<const char *>(ptr);
        auto after = blocks.upper_bound(at);
        if (after == blocks.begin()) return nullptr;
        const TensorBlock &block = (--after)->second;
        return at < after->first + block.capacity ? &block : nullptr;
    }
    std::deque<TensorBlock *> &idle_of(size_t capacity) { return idle[__builtin_ctzll(capacity / kTensorSmallest)]; }
    // Makes `most` of what is held, of the longest idle blocks: the caller frees what it is given.
    void shrink(size_t most, std::vector<void *> &doomed)
    {
        while (held > most) {
            std::deque<TensorBlock *> *oldest = nullptr;
            for (auto &blocks_of_size : idle)
                if (!blocks_of_size.empty() && (oldest == nullptr || blocks_of_size.front()->idle_since < oldest->front()->idle_since)) oldest = &blocks_of_size;
            const TensorBlock *const block = oldest->front();
            oldest->pop_front();
            held -= block->capacity;
            doomed.push_back(block->ptr);
            blocks.erase(static_cast<const char *>(doomed.back()));
        }
    }
};
TensorPool &tensor_pool()  // never destroyed: tensors may be freed while the process is shutting down
{
    static TensorPool *pool = new TensorPool;
    return *pool;
}
size_t tensor_capacity(size_t bytes)
{
    size_t capacity = kTensorSmallest;
    while (capacity < bytes) capacity *= 2;
    return capacity;
}
void tensor_release_idle()
{
    std::vector<void *> doomed;
    {
        TensorPool &pool = tensor_pool();
        std::lock_guard<std::mutex> lock(pool.mutex);
        pool.shrink(0, doomed);
    }
    for (void *ptr : doomed) (void)hipFree(ptr);
}

// Where `bytes` from `ptr` on lie.  What is behind a tensor in its block is not the tensor's, and an idle block is nobody's: a copy there
// is refused as the runtime refuses one that passes an allocation's end.
enum class TensorRange { kElsewhere, kInside, kOutside };
TensorRange tensor_range(const void *ptr, size_t bytes, int *device)
{
    TensorPool &pool = tensor_pool();
    std::lock_guard<std::mutex> lock(pool.mutex);
    const TensorBlock *block = pool.find(ptr);
    if (block == nullptr) return TensorRange::kElsewhere;
    *device = block->device;
    const size_t offset = static_cast<size_t>(static_cast<const char *>(ptr) - static_cast<const char *>(block->ptr));
    return block->idle_since == 0 && offset <= block->bytes && bytes <= block->bytes - offset ? TensorRange::kInside : TensorRange::kOutside;
}
bool passes_tensor_end(const void *ptr, size_t bytes)
{
    int device;
    return tensor_range(ptr, bytes, &device) == TensorRange::kOutside;
}

// Whether a kernel on `stream` may access `bytes` from `ptr` on: memory of the current device, which is the stream's as well, all of it in
// one allocation.  Whatever else is left to the runtime's copy, which takes or refuses it.
bool kernel_may_access(const void *ptr, size_t bytes, hipStream_t stream)
{
    int current = 0, device = 0, streams = 0;
    if (hipGetDevice(&current) != hipSuccess || (stream != nullptr && hipStreamGetDevice(stream, &streams) != hipSuccess)) {
        (void)hipGetLastError();
        return false;
    }
    if (stream != nullptr && streams != current) return false;
    const TensorRange range = tensor_range(ptr, bytes, &device);
    if (range != TensorRange::kElsewhere) return range == TensorRange::kInside && device == current;
    hipPointerAttribute_t attributes;
    if (hipPointerGetAttributes(&attributes, ptr) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    if (attributes.type != hipMemoryTypeDevice || attributes.device != current) return false;
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    if (hipMemGetAddressRange(&base, &size, const_cast<void *>(ptr)) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    const size_t offset = static_cast<size_t>(static_cast<const char *>(ptr) - static_cast<const char *>(base));
    return offset <= size && bytes <= size - offset;
}
}  // namespace

hipError_t device_malloc(void **out, size_t bytes)
{
    hipError_t rc = hipMalloc(out, bytes);
    if (rc == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        tensor_release_idle();
        rc = hipMalloc(out, bytes);
    }
    return rc;
}

namespace {
// Scratch is keyed by (stream, host thread, slot): launches on one stream from one thread are ordered, so they never
// use the buffer at the same time; two host threads that share a stream (every caller that passes none shares the
// NULL stream) each get a buffer of their own, so one thread growing its scratch can never free memory that a
// kernel the other thread has just been handed is about to use.
//
// Lifetime: an entry lives until its stream is destroyed (st_hip_stream_destroy) or st_hip_release_scratch is called
// for the stream.  When its host thread exits, the entry is not freed (kernels of that thread may still be queued) but
// orphaned, and the next thread that asks for scratch on that stream and slot adopts it: work on one stream is
// ordered and the former owner can no longer be between receiving the pointer and launching, so a pool of short-lived
// threads keeps re-using the same few buffers instead of leaking one per thread.
//
// Capture: a launch recorded into a graph keeps the buffer it was handed.  Such a buffer is never freed by growing past it
// (the graph may be replayed later): it is kept beside the entries, and freed with them.
struct WorkspaceEntry {
    hipStream_t stream;
    std::thread::id owner;  // std::thread::id() once the owning thread has exited
    void *ptr;
    size_t capacity;
    int slot;
    bool growing;  // its owner is replacing the buffer outside the lock
    bool captured;  // handed out while the stream was being captured
};
struct RetiredBuffer {
    hipStream_t stream;
    void *ptr;
};
// Never destroyed: threads may exit (and orphan their entries) while the process is shutting down.
std::mutex &workspace_mutex()
{
    static std::mutex *mutex = new std::mutex;
    return *mutex;
}
std::vector<WorkspaceEntry> &workspace_entries()
{
    static std::vector<WorkspaceEntry> *entries = new std::vector<WorkspaceEntry>;
    return *entries;
}
std::vector<RetiredBuffer> &retired_buffers()
{
    static std::vector<RetiredBuffer> *buffers = new std::vector<RetiredBuffer>;
    return *buffers;
}

struct ThreadScratchGuard {
    bool armed = false;
    ~ThreadScratchGuard()
    {
        if (!armed) return;
        const std::thread::id me = std::this_thread::get_id();
        std::lock_guard<std::mutex> lock(workspace_mutex());
        for (WorkspaceEntry &e : workspace_entries())
            if (e.owner == me) e.owner = std::thread::id();
    }
};
thread_local ThreadScratchGuard thread_scratch_guard;

bool being_captured(hipStream_t stream)
{
    if (stream == nullptr) return false;  // the legacy stream cannot be captured
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(stream, &status) == hipSuccess && status != hipStreamCaptureStatusNone;
}

// An allocation is no part of a graph, and allowed during a capture of any mode only where the thread says that it means it.
hipError_t scratch_malloc(void **out, size_t bytes, bool capturing)
{
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    if (capturing && hipThreadExchangeStreamCaptureMode(&mode) != hipSuccess) return hipErrorStreamCaptureUnsupported;
    const hipError_t rc = capturing ? hipMalloc(out, bytes) : device_malloc(out, bytes);
    if (rc != hipSuccess) (void)hipGetLastError();  // the caller may go on without scratch
    if (capturing) (void)hipThreadExchangeStreamCaptureMode(&mode);
    return rc;
}

WorkspaceEntry *find_entry(hipStream_t stream, std::thread::id owner, int slot)
{
    for (WorkspaceEntry &e : workspace_entries())
        if (e.stream == stream && e.owner == owner && e.slot == slot) return &e;
    return nullptr;
}
}  // namespace

hipError_t stream_workspace(hipStream_t stream, size_t bytes, void **out) { return stream_workspace_slot(stream, 0, bytes, out); }

hipError_t stream_workspace_slot(hipStream_t stream, int slot, size_t bytes, void **out)
{
    const std::thread::id me = std::this_thread::get_id();
    const size_t wanted = bytes ? bytes : 256;
    const bool capturing = being_captured(stream);
    void *old = nullptr;
    {
        std::lock_guard<std::mutex> lock(workspace_mutex());
        thread_scratch_guard.armed = true;
        WorkspaceEntry *e = find_entry(stream, me, slot);
        if (!e) {
            e = find_entry(stream, std::thread::id(), slot);  // a buffer whose thread has exited
            if (e) e->owner = me;
        }
        if (e) {
            if (e->ptr != nullptr && e->capacity >= wanted) {
                e->captured |= capturing;
                *out = e->ptr;
                return hipSuccess;
            }
            // (launches recorded earlier in this capture may hold the buffer as well)
            if (e->ptr != nullptr && (e->captured || capturing)) {
                retired_buffers().push_back(RetiredBuffer{stream, e->ptr});
                e->ptr = nullptr;
            }
            // Grow: outside the lock (the wait for the stream must not stall other threads' launches).  The entry stays
            // in the table, owned by this thread and empty, so nobody else touches it meanwhile.
            old = e->ptr;
            e->ptr = nullptr;
            e->capacity = 0;
            e->captured = false;
            e->growing = true;
        }
    }
    if (old) {
        // earlier launches on this stream may still be using the old buffer
        hipError_t rc = hipStreamSynchronize(stream);
        if (rc == hipSuccess) rc = hipFree(old);
        if (rc != hipSuccess) {
            std::lock_guard<std::mutex> lock(workspace_mutex());
            if (WorkspaceEntry *e = find_entry(stream, me, slot)) e->growing = false;
            return rc;
        }
    }
    void *fresh = nullptr;
    const hipError_t rc = scratch_malloc(&fresh, wanted, capturing);
    std::lock_guard<std::mutex> lock(workspace_mutex());
    WorkspaceEntry *e = find_entry(stream, me, slot);
    if (rc != hipSuccess) {
        if (e) e->growing = false;
        return rc;
    }
    if (e) {
        e->ptr = fresh;
        e->capacity = wanted;
        e->growing = false;
        e->captured = capturing;
    } else {
        workspace_entries().push_back(WorkspaceEntry{stream, me, fresh, wanted, slot, false, capturing});
    }
    *out = fresh;
    return hipSuccess;
}

// Called after the stream has been drained (before it is destroyed, or by st_hip_release_scratch).
void release_stream_workspace(hipStream_t stream)
{
    std::vector<void *> doomed;
    {
        std::lock_guard<std::mutex> lock(workspace_mutex());
        std::vector<WorkspaceEntry> &entries = workspace_entries();
        for (size_t i = entries.size(); i-- > 0;) {
            if (entries[i].stream != stream || entries[i].growing) continue;
            if (entries[i].ptr) doomed.push_back(entries[i].ptr);
            entries.erase(entries.begin() + static_cast<long>(i));
        }
        std::vector<RetiredBuffer> &retired = retired_buffers();
        for (size_t i = retired.size(); i-- > 0;) {
            if (retired[i].stream != stream) continue;
            doomed.push_back(retired[i].ptr);
            retired.erase(retired.begin() + static_cast<long>(i));
        }
    }
    for (void *ptr : doomed) (void)hipFree(ptr);
}

size_t stream_workspace_entry_count()
{
    std::lock_guard<std::mutex> lock(workspace_mutex());
    return workspace_entries().size() + retired_buffers().size();
}

}  // namespace sthip

using namespace sthip;

extern "C" {

int st_hip_init(void) { return ensure_init(); }

int st_hip_real_backend_compiled(void) { return 1; }

int st_hip_device_count(void)
{
    if (ensure_init() != ST_HIP_OK) return 0;
    return static_cast<int>(runtime().devices.size());
}

int st_hip_device_name(int index, char *buf, size_t len)
{
    ST_HIP_CHECK(ensure_init());
    if (index < 0 || static_cast<size_t>(index) >= runtime().devices.size() || !buf || len == 0)
        return fail(ST_HIP_ERR_INVALID, "device index %d out of range", index);
    const hipDeviceProp_t &p = runtime().devices[static_cast<size_t>(index)];
    snprintf(buf, len, "%s", p.name[0] ? p.name : p.gcnArchName);
    return ST_HIP_OK;
}

int st_hip_device_properties(int index, st_hip_device_props *out)
{
    ST_HIP_CHECK(ensure_init());
    if (index < 0 || static_cast<size_t>(index) >= runtime().devices.size() || !out)
        return fail(ST_HIP_ERR_INVALID, "device index %d out of range", index);
    const hipDeviceProp_t &p = runtime().devices[static_cast<size_t>(index)];
    std::memset(out, 0, sizeof *out);
    out->compute_units = p.multiProcessorCount;
    out->clock_khz = p.clockRate;
    out->memory_clock_khz = p.memoryClockRate;
    out->memory_bus_bits = p.memoryBusWidth;
    out->wavefront_size = p.warpSize;
    out->lds_bytes_per_block = static_cast<int>(p.sharedMemPerBlock);
    out->l2_bytes = p.l2CacheSize;
    out->total_memory_bytes = p.totalGlobalMem;
    snprintf(out->arch, sizeof out->arch, "%s", p.gcnArchName);
    return ST_HIP_OK;
}

int st_hip_probe(st_hip_probe_result *out)
{
    if (!out) return fail(ST_HIP_ERR_INVALID, "st_hip_probe received a null out-pointer");
    std::memset(out, 0, sizeof *out);
    int count = 0;
    const hipError_t rc = hipGetDeviceCount(&count);
    if (rc != hipSuccess) (void)hipGetLastError();
    out->available = rc == hipSuccess && count > 0;
    out->device_count = rc == hipSuccess ? count : 0;
    if (ensure_init() == ST_HIP_OK) {
        out->initialized = 1;
    } else {
        snprintf(out->error, sizeof out->error, "%s", g_last_error.c_str());
    }
    return ST_HIP_OK;
}

size_t st_hip_last_error_message(char *buf, size_t len)
{
    if (buf && len > 0) snprintf(buf, len, "%s", g_last_error.c_str());
    return g_last_error.size();
}

int st_hip_malloc(void **device_ptr, size_t bytes)
{
    ST_HIP_CHECK(ensure_init());
    if (!device_ptr) return fail(ST_HIP_ERR_INVALID, "st_hip_malloc received a null out-pointer");
    *device_ptr = nullptr;
    ST_HIP_TRY(device_malloc(device_ptr, bytes ? bytes : 1), "hipMalloc");  // real.rs:652 max(1)
    return ST_HIP_OK;
}

int st_hip_free(void *device_ptr)
{
    if (!device_ptr) return ST_HIP_OK;
    {
        TensorPool &pool = tensor_pool();
        std::lock_guard<std::mutex> lock(pool.mutex);
        const auto found = pool.blocks.find(static_cast<const char *>(device_ptr));
        if (found != pool.blocks.end()) {
            if (found->second.idle_since != 0) return hip_fail(hipErrorInvalidValue, "hipFree");  // freed before
            pool.blocks.erase(found);  // (the address may come back as something else)
        }
    }
    ST_HIP_TRY(hipFree(device_ptr), "hipFree");
    return ST_HIP_OK;
}

int st_hip_tensor_malloc(void **device_ptr, size_t bytes)
{
    ST_HIP_CHECK(ensure_init());
    if (!device_ptr) return fail(ST_HIP_ERR_INVALID, "st_hip_tensor_malloc received a null out-pointer");
    *device_ptr = nullptr;
    if (bytes > kTensorLargest) return st_hip_malloc(device_ptr, bytes);
    const size_t capacity = tensor_capacity(bytes);
    int device = 0;
    ST_HIP_TRY(hipGetDevice(&device), "hipGetDevice");
    {
        TensorPool &pool = tensor_pool();
        std::lock_guard<std::mutex> lock(pool.mutex);
        std::deque<TensorBlock *> &idle = pool.idle_of(capacity);
        for (size_t i = idle.size(); i-- > 0;) {
            TensorBlock &block = *idle[i];
            if (block.device != device) continue;
            idle.erase(idle.begin() + static_cast<long>(i));
            *device_ptr = block.ptr;
            block.bytes = bytes;
            block.idle_since = 0;
            pool.held -= capacity;
            return ST_HIP_OK;
        }
    }
    ST_HIP_TRY(device_malloc(device_ptr, capacity), "hipMalloc");
    TensorPool &pool = tensor_pool();
    std::lock_guard<std::mutex> lock(pool.mutex);
    pool.blocks[static_cast<const char *>(*device_ptr)] = TensorBlock{*device_ptr, capacity, bytes, device, 0};
    return ST_HIP_OK;
}

int st_hip_tensor_free(void *device_ptr, size_t bytes)
{
    if (!device_ptr) return ST_HIP_OK;
    std::vector<void *> doomed;
    auto keep = [&] {
        TensorPool &pool = tensor_pool();
        std::lock_guard<std::mutex> lock(pool.mutex);
        const auto found = pool.blocks.find(static_cast<const char *>(device_ptr));
        if (found == pool.blocks.end() || found->second.idle_since != 0 || bytes > kTensorLargest) return false;
        TensorBlock &block = found->second;
        pool.held += block.capacity;
        pool.shrink(kTensorMost, doomed);
        block.idle_since = ++pool.frees;
        pool.idle_of(block.capacity).push_back(&block);
        return true;
    };
    if (!keep()) return st_hip_free(device_ptr);
    for (void *ptr : doomed) (void)hipFree(ptr);
    return ST_HIP_OK;
}

int st_hip_tensor_upload(void *device_ptr, const void *host_src, size_t bytes)
{
    PinnedBuffer stage;
    const size_t groups = (bytes + kUploadGroup - 1) / kUploadGroup, words_at = (bytes + 15) / 16 * 16;
    if (bytes == 0 || bytes > kUploadMost || reinterpret_cast<uintptr_t>(device_ptr) % 16 != 0 || host_memory(host_src) != HostMemory::kOrdinary ||
        !kernel_may_access(device_ptr, bytes, nullptr) || !pinned_acquire(words_at + groups * sizeof(unsigned), &stage))
        return st_hip_memcpy_h2d(device_ptr, host_src, bytes, nullptr);
    count_transfer(true, bytes);
    unsigned *const read = reinterpret_cast<unsigned *>(static_cast<unsigned char *>(stage.ptr) + words_at);
    std::memcpy(stage.ptr, host_src, bytes);
    std::memset(read, 0, groups * sizeof(unsigned));
    const hipError_t rc = launch_copy_from_pinned(device_ptr, stage.ptr, bytes, nullptr, read);
    if (rc != hipSuccess) {
        pinned_release(stage);
        return hip_fail(rc, "copy launch");
    }
    pinned_release_when_read(stage, read, groups);
    return ST_HIP_OK;
}

int st_hip_memcpy_h2d(void *device_dst, const void *host_src, size_t bytes, void *stream)
{
    if (bytes == 0) return ST_HIP_OK;
    if (passes_tensor_end(device_dst, bytes)) return hip_fail(hipErrorInvalidValue, "hipMemcpyAsync(H2D)");
    count_transfer(true, bytes);
    ST_HIP_TRY(hipMemcpyAsync(device_dst, host_src, bytes, hipMemcpyHostToDevice, as_stream(stream)),
               "hipMemcpyAsync(H2D)");
    ST_HIP_TRY(hipStreamSynchronize(as_stream(stream)), "hipStreamSynchronize");
    return ST_HIP_OK;
}

int st_hip_memcpy_d2h(void *host_dst, const void *device_src, size_t bytes, void *stream)
{
    if (bytes == 0) return ST_HIP_OK;
    if (passes_tensor_end(device_src, bytes)) return hip_fail(hipErrorInvalidValue, "hipMemcpyAsync(D2H)");
    count_transfer(false, bytes);
    PinnedBuffer stage;
    const bool staged = bytes <= kReadMost && host_memory(host_dst) == HostMemory::kOrdinary && pinned_acquire(bytes, &stage);
    if (staged && reinterpret_cast<uintptr_t>(device_src) % 16 == 0 && kernel_may_access(device_src, bytes, as_stream(stream))) {
        const size_t pieces = (bytes + kCopyPiece - 1) / kCopyPiece;
        unsigned *const words = stage.words();
        std::memset(words, 0, pieces * sizeof(unsigned));
        hipError_t rc = launch_copy_to_pinned(stage.ptr, device_src, bytes, words, as_stream(stream));
        const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(1);
        bool waited = rc != hipSuccess;
        for (size_t p = 0; rc == hipSuccess && p < pieces;) {
            if (__atomic_load_n(&words[p], __ATOMIC_ACQUIRE) != 0) {
                const size_t at = p * kCopyPiece;
                std::memcpy(static_cast<unsigned char *>(host_dst) + at, static_cast<const unsigned char *>(stage.ptr) + at, std::min(kCopyPiece, bytes - at));
                ++p;
            } else if (waited) {
                rc = hipErrorUnknown;
            } else if (std::chrono::steady_clock::now() > until) {
                rc = hipStreamSynchronize(as_stream(stream));
                waited = true;
            }
        }
        pinned_release(stage);
        ST_HIP_TRY(rc, "copy to the host");
        return ST_HIP_OK;
    }
    const hipError_t rc = hipMemcpyAsync(staged ? stage.ptr : host_dst, device_src, bytes, hipMemcpyDeviceToHost, as_stream(stream));
    const hipError_t drained = hipStreamSynchronize(as_stream(stream));  // before the pinned memory is handed back
    if (staged && rc == hipSuccess && drained == hipSuccess) std::memcpy(host_dst, stage.ptr, bytes);
    pinned_release(stage);
    ST_HIP_TRY(rc, "hipMemcpyAsync(D2H)");
    ST_HIP_TRY(drained, "hipStreamSynchronize");
    return ST_HIP_OK;
}

int st_hip_memset_zero(void *device_dst, size_t bytes, void *stream)
{
    if (bytes == 0) return ST_HIP_OK;
    if (passes_tensor_end(device_dst, bytes)) return hip_fail(hipErrorInvalidValue, "hipMemsetAsync");
    ST_HIP_TRY(hipMemsetAsync(device_dst, 0, bytes, as_stream(stream)), "hipMemsetAsync");
    return ST_HIP_OK;
}

int st_hip_transfer_counters(uint64_t counters[4], int reset)
{
    if (!counters) return fail(ST_HIP_ERR_INVALID, "st_hip_transfer_counters received a null out-pointer");
    for (int i = 0; i < 4; ++i)
        counters[i] = reset ? g_transfers[i].exchange(0, std::memory_order_relaxed) : g_transfers[i].load(std::memory_order_relaxed);
    return ST_HIP_OK;
}

int st_hip_stream_create(void **stream)
{
    ST_HIP_CHECK(ensure_init());
    if (!stream) return fail(ST_HIP_ERR_INVALID, "st_hip_stream_create received a null out-pointer");
    hipStream_t raw = nullptr;
    ST_HIP_TRY(hipStreamCreate(&raw), "hipStreamCreate");
    *stream = raw;
    return ST_HIP_OK;
}

int st_hip_stream_synchronize(void *stream)
{
    ST_HIP_TRY(hipStreamSynchronize(as_stream(stream)), "hipStreamSynchronize");
    return ST_HIP_OK;
}

int st_hip_stream_destroy(void *stream)
{
    if (!stream) return ST_HIP_OK;
    // Same order as HipStream::drop (real.rs:207-214): drain, then release.
    (void)hipStreamSynchronize(as_stream(stream));
    release_stream_workspace(as_stream(stream));
    ST_HIP_TRY(hipStreamDestroy(as_stream(stream)), "hipStreamDestroy");
    return ST_HIP_OK;
}

int st_hip_release_scratch(void *stream)
{
    ST_HIP_CHECK(ensure_init());
    ST_HIP_TRY(hipStreamSynchronize(as_stream(stream)), "hipStreamSynchronize");
    release_stream_workspace(as_stream(stream));
    pinned_release_idle();
    if (stream == nullptr) tensor_release_idle();
    return ST_HIP_OK;
}

size_t st_hip_scratch_buffer_count(void) { return stream_workspace_entry_count(); }

int st_hip_pinned_memory_counters(uint64_t *counters)
{
    if (!counters) return fail(ST_HIP_ERR_INVALID, "pinned_memory_counters received a null out-pointer");
    PinnedPool &pool = pinned_pool();
    std::lock_guard<std::mutex> lock(pool.mutex);
    counters[0] = pool.held;
    counters[1] = pool.allocations;
    return ST_HIP_OK;
}

int st_hip_device_synchronize(void)
{
    ST_HIP_TRY(hipDeviceSynchronize(), "hipDeviceSynchronize");
    return ST_HIP_OK;
}

int st_hip_event_create(void **event)
{
    ST_HIP_CHECK(ensure_init());
    if (!event) return fail(ST_HIP_ERR_INVALID, "st_hip_event_create received a null out-pointer");
    hipEvent_t raw = nullptr;
    ST_HIP_TRY(hipEventCreate(&raw), "hipEventCreate");
    *event = raw;
    return ST_HIP_OK;
}

int st_hip_event_record(void *event, void *stream)
{
    ST_HIP_TRY(hipEventRecord(static_cast<hipEvent_t>(event), as_stream(stream)), "hipEventRecord");
    return ST_HIP_OK;
}

int st_hip_event_synchronize(void *event)
{
    ST_HIP_TRY(hipEventSynchronize(static_cast<hipEvent_t>(event)), "hipEventSynchronize");
    return ST_HIP_OK;
}

int st_hip_event_elapsed_ms(void *start, void *stop, float *milliseconds)
{
    if (!milliseconds) return fail(ST_HIP_ERR_INVALID, "st_hip_event_elapsed_ms received a null out-pointer");
    ST_HIP_TRY(hipEventElapsedTime(milliseconds, static_cast<hipEvent_t>(start), static_cast<hipEvent_t>(stop)),
               "hipEventElapsedTime");
    return ST_HIP_OK;
}

int st_hip_event_destroy(void *event)
{
    if (!event) return ST_HIP_OK;
    ST_HIP_TRY(hipEventDestroy(static_cast<hipEvent_t>(event)), "hipEventDestroy");
    return ST_HIP_OK;
}

}  // extern "C"
