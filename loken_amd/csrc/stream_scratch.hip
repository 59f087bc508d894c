#include "stream_scratch.h"

#include <thread>

namespace {

struct Entry {
    hipStream_t stream;
    std::thread::id thread;   // hipStreamPerThread is one handle for a stream of every thread
    std::shared_ptr<LkStreamScratch> scratch;
};
std::mutex g_mu;
std::vector<Entry>& g_entries = *new std::vector<Entry>;   // never destroyed: the process may end after its runtime
unsigned long long g_clock = 0;

}  // namespace

struct LkStreamScratch::Block {
    int device;
    LkScratchUse use;
    void* ptr;
    size_t size;
    ~Block() {   // hipFree waits for the device
        int current = 0;
        if (hipGetDevice(&current) == hipSuccess && hipSetDevice(device) == hipSuccess) {
            (void)hipFree(ptr);
            (void)hipSetDevice(current);
        }
        (void)hipGetLastError();
    }
};

std::vector<std::weak_ptr<LkStreamScratch::Block>>& LkStreamScratch::blocks() {
    static auto& all = *new std::vector<std::weak_ptr<Block>>;
    return all;
}

void LkStreamScratch::free_all() {
    for (auto& b : now_) b.reset();
    kept_.clear();
}

void* LkStreamScratch::get(LkScratchUse use, size_t bytes, hipStream_t stream) {
    std::shared_ptr<Block>& own = now_[use];
    const bool fits = own && own->size >= bytes;
    if (fits && recorded) return own->ptr;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cs) != hipSuccess) (void)hipGetLastError();
    if (cs != hipStreamCaptureStatusNone) recorded = true;
    if (fits) return own->ptr;
    if (cs != hipStreamCaptureStatusNone) {
        std::lock_guard<std::mutex> lock(g_mu);
        for (auto it = blocks().rbegin(); it != blocks().rend(); ++it)
            if (auto b = it->lock(); b && b->device == device_ && b->use == use && b->size >= bytes) {
                kept_.push_back(b);   // for the graph; calls of this stream outside it get their own
                return b->ptr;
            }
        return nullptr;
    }
    void* fresh = nullptr;
    const size_t want = (bytes + bytes / 4 + 255) & ~(size_t)255;
    if (hipMalloc(&fresh, want) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    if (own) kept_.push_back(own);
    own = std::shared_ptr<Block>(new Block{device_, use, fresh, want});
    std::lock_guard<std::mutex> lock(g_mu);
    auto& all = blocks();
    for (size_t i = 0; i < all.size();) {
        if (all[i].expired()) all.erase(all.begin() + (long)i);
        else ++i;
    }
    all.push_back(own);
    return fresh;
}

std::shared_ptr<LkStreamScratch> lk_stream_scratch(hipStream_t stream) {
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) (void)hipGetLastError();
    const std::thread::id thread = stream == hipStreamPerThread ? std::this_thread::get_id() : std::thread::id();
    std::shared_ptr<LkStreamScratch> given_up;   // freed after the lock
    std::lock_guard<std::mutex> lock(g_mu);
    int held = 0;
    size_t oldest = g_entries.size();
    for (size_t i = 0; i < g_entries.size(); ++i) {
        Entry& e = g_entries[i];
        if (e.scratch->device() != device) continue;
        if (e.stream == stream && e.thread == thread) {
            e.scratch->used_at = ++g_clock;
            return e.scratch;
        }
        if (e.scratch->recorded) continue;
        ++held;
        if (oldest == g_entries.size() || e.scratch->used_at < g_entries[oldest].scratch->used_at) oldest = i;
    }
    if (held >= LK_SCRATCH_STREAMS) {
        given_up = std::move(g_entries[oldest].scratch);
        g_entries.erase(g_entries.begin() + (long)oldest);
    }
    g_entries.push_back(Entry{stream, thread, std::make_shared<LkStreamScratch>(device)});
    g_entries.back().scratch->used_at = ++g_clock;
    return g_entries.back().scratch;
}

void lk_stream_scratch_release(int device) {
    int current = 0;
    if (hipGetDevice(&current) != hipSuccess) { (void)hipGetLastError(); return; }
    std::vector<Entry> entries;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        for (size_t i = 0; i < g_entries.size();) {
            if (device >= 0 && g_entries[i].scratch->device() != device) { ++i; continue; }
            entries.push_back(std::move(g_entries[i]));
            g_entries.erase(g_entries.begin() + (long)i);
        }
    }
    for (Entry& e : entries) {
        std::lock_guard<std::recursive_mutex> lock(e.scratch->mu);
        if (hipSetDevice(e.scratch->device()) != hipSuccess) { (void)hipGetLastError(); continue; }
        (void)hipDeviceSynchronize();   // queued kernels may still read what is freed below
        e.scratch->free_all();
    }
    (void)hipSetDevice(current);
    (void)hipGetLastError();
}
