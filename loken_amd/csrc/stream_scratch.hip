#include "stream_scratch.h"

#include <thread>
#include <utility>
#include <vector>

namespace {

struct Block {
    void* ptr = nullptr;
    size_t size = 0;
    LkScratchUse use = LK_SCRATCH_USES;
};
constexpr unsigned EVERY_USE = (1u << LK_SCRATCH_USES) - 1;

// Who a pool belongs to: a stream, what a stream records in one capture, or (`shared`) the streams without their own.
struct Owner {
    int device = 0;
    hipStream_t stream = nullptr;
    std::thread::id thread;   // hipStreamPerThread is one handle for a stream of every thread
    bool recording = false, shared = false;
    unsigned long long capture = 0;
    bool operator==(const Owner& o) const {
        return device == o.device && stream == o.stream && thread == o.thread && recording == o.recording && shared == o.shared &&
               capture == o.capture;
    }
};

std::mutex g_mu;   // of what follows; taken inside a pool's lock, never around one
std::vector<std::shared_ptr<LkScratchPool>>& g_streams = *new std::vector<std::shared_ptr<LkScratchPool>>;   // never destroyed: the
std::vector<std::shared_ptr<LkScratchPool>>& g_graphs = *new std::vector<std::shared_ptr<LkScratchPool>>;    // process may end after its runtime
std::vector<int>& g_tickets = *new std::vector<int>;   // given back
int g_next_ticket = 0;

}  // namespace

struct LkScratchPool {
    explicit LkScratchPool(const Owner& o) : owner(o) {   // caller holds g_mu
        if (o.recording) return;
        if (!g_tickets.empty()) {
            ticket = g_tickets.back();
            g_tickets.pop_back();
        } else if (g_next_ticket < LK_SCRATCH_TICKETS) {
            ticket = g_next_ticket++;
        }
    }
    ~LkScratchPool() {   // its kernels are over: a pool leaves the tables after the device was waited for
        free_blocks(take_blocks(EVERY_USE));
        if (last_use && hipEventDestroy(last_use) != hipSuccess) (void)hipGetLastError();
        std::lock_guard<std::mutex> lock(g_mu);
        if (ticket >= 0) g_tickets.push_back(ticket);
    }

    std::vector<Block> take_blocks(unsigned uses) {   // caller holds mu and g_mu, or has the last reference
        std::vector<Block> taken, stay;
        for (const Block& b : kept) (uses >> b.use & 1 ? taken : stay).push_back(b);
        kept = std::move(stay);
        for (Block& b : now)
            if (b.ptr && uses >> b.use & 1) {
                taken.push_back(b);
                b = Block{};
            }
        return taken;
    }
    bool empty() const {
        for (const Block& b : now)
            if (b.ptr) return false;
        return kept.empty();
    }
    void free_blocks(const std::vector<Block>& blocks) const {   // hipFree waits for the device
        int current = 0;
        if (blocks.empty() || hipGetDevice(&current) != hipSuccess || hipSetDevice(owner.device) != hipSuccess) return;
        for (const Block& b : blocks) (void)hipFree(b.ptr);
        (void)hipSetDevice(current);
        (void)hipGetLastError();
    }

    const Owner owner;
    int ticket = -1;
    std::recursive_mutex mu;
    bool retired = false;   // out of the table: the stream's next call gets another one
    // written under mu and g_mu, so either is enough to read
    Block now[LK_SCRATCH_USES];
    std::vector<Block> kept;   // outgrown and not freed
    // of a shared pool, under mu: how many of the thread's launchers hold it, whether they took a buffer, and the
    // last kernels of those before them
    int held = 0;
    bool taken = false;
    hipEvent_t last_use = nullptr;
};

namespace {

Owner owner_of(hipStream_t stream) {
    Owner o;
    if (hipGetDevice(&o.device) != hipSuccess) (void)hipGetLastError();
    o.stream = stream;
    if (stream == hipStreamPerThread) o.thread = std::this_thread::get_id();
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    unsigned long long id = 0;
    if (hipStreamGetCaptureInfo(stream, &status, &id) != hipSuccess) {
        (void)hipGetLastError();
        status = hipStreamCaptureStatusNone;
    }
    if (status != hipStreamCaptureStatusNone) {
        o.recording = true;
        o.capture = id;
    }
    return o;
}

std::shared_ptr<LkScratchPool> pool_of(Owner owner) {
    std::lock_guard<std::mutex> lock(g_mu);
    auto& pools = owner.recording ? g_graphs : g_streams;
    int of_device = 0;
    std::shared_ptr<LkScratchPool> shared;
    for (size_t i = pools.size(); i-- > 0;) {   // a capture's pool is among the last
        if (pools[i]->owner == owner) return pools[i];
        if (pools[i]->owner.device != owner.device) continue;
        if (pools[i]->owner.shared) shared = pools[i];
        else ++of_device;
    }
    if (!owner.recording && of_device >= LK_SCRATCH_STREAMS) {
        if (shared) return shared;
        const int device = owner.device;
        owner = Owner{};
        owner.device = device;
        owner.shared = true;
    }
    pools.push_back(std::make_shared<LkScratchPool>(owner));
    return pools.back();
}

// Whether a call outside any capture has reserved `bytes` for `use`, and the device's graphs have room for `want` more.
bool graph_may_hold(int device, LkScratchUse use, size_t bytes, size_t want) {
    std::lock_guard<std::mutex> lock(g_mu);
    bool reserved = false;
    for (const auto& p : g_streams) reserved = reserved || (p->owner.device == device && p->now[use].size >= bytes);
    size_t held = 0;
    for (const auto& p : g_graphs) {
        if (p->owner.device != device) continue;
        for (const Block& b : p->now) held += b.size;
        for (const Block& b : p->kept) held += b.size;
    }
    return reserved && want <= LK_SCRATCH_GRAPH_BYTES && held <= LK_SCRATCH_GRAPH_BYTES - want;
}

// Allocating and freeing are no operations of a stream and no part of a graph; in the relaxed mode they are allowed
// whatever streams are recording, this one or another thread's.
class RelaxedCapture {
  public:
    RelaxedCapture() : switched_(hipThreadExchangeStreamCaptureMode(&mode_) == hipSuccess) {}
    ~RelaxedCapture() {
        if (switched_) (void)hipThreadExchangeStreamCaptureMode(&mode_);
        (void)hipGetLastError();
    }

  private:
    hipStreamCaptureMode mode_ = hipStreamCaptureModeRelaxed;
    const bool switched_;
};

}  // namespace

LkScratch::LkScratch(hipStream_t stream) : stream_(stream) {
    const Owner owner = owner_of(stream);
    do {
        pool_ = pool_of(owner);
        lock_ = std::unique_lock<std::recursive_mutex>(pool_->mu);
        if (!pool_->retired) break;
        lock_.unlock();
    } while (true);
    ++pool_->held;
}

LkScratch::~LkScratch() {
    LkScratchPool& pool = *pool_;
    if (--pool.held > 0 || !pool.taken) return;
    pool.taken = false;   // (set by a shared pool only)
    if (!pool.last_use && hipEventCreateWithFlags(&pool.last_use, hipEventDisableTiming) != hipSuccess) pool.last_use = nullptr;
    if (!pool.last_use || hipEventRecord(pool.last_use, stream_) != hipSuccess) (void)hipStreamSynchronize(stream_);
    (void)hipGetLastError();
}

void* LkScratch::get(LkScratchUse use, size_t bytes) {
    LkScratchPool& pool = *pool_;
    if (pool.owner.shared && !pool.taken) {
        if (pool.last_use && hipStreamWaitEvent(stream_, pool.last_use, 0) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        pool.taken = true;
    }
    Block& own = pool.now[use];
    if (own.ptr && own.size >= bytes) return own.ptr;
    const size_t want = ((use == LK_SCRATCH_FIXUP ? bytes : bytes + bytes / 4) + 255) & ~(size_t)255;   // (fixup: one size)
    if (pool.owner.recording && !graph_may_hold(pool.owner.device, use, bytes, want)) return nullptr;
    RelaxedCapture relaxed;
    if (own.ptr) {
        // Outgrown. Kernels of this stream that still use it are waited for by hipFree; a graph's nodes keep theirs.
        Block outgrown = own;
        const bool freed = !pool.owner.recording && hipFree(outgrown.ptr) == hipSuccess;
        std::lock_guard<std::mutex> lock(g_mu);
        own = Block{};
        if (!freed) pool.kept.push_back(outgrown);
    }
    void* fresh = nullptr;
    if (hipMalloc(&fresh, want) != hipSuccess) return nullptr;
    std::lock_guard<std::mutex> lock(g_mu);
    own = Block{fresh, want, use};
    return fresh;
}

int LkScratch::ticket() const { return pool_->ticket; }

bool LkScratch::recording() const { return pool_->owner.recording; }

void lk_stream_scratch_release(int device, unsigned uses) {
    int current = 0;
    if (hipGetDevice(&current) != hipSuccess) { (void)hipGetLastError(); return; }
    std::vector<std::shared_ptr<LkScratchPool>> pools;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        for (auto* list : {&g_streams, &g_graphs})
            for (const auto& p : *list)
                if (device < 0 || p->owner.device == device) pools.push_back(p);
    }
    for (auto& p : pools) {
        std::lock_guard<std::recursive_mutex> lock(p->mu);
        // queued kernels may still read what is freed: nothing is where they cannot be waited for
        if (hipSetDevice(p->owner.device) != hipSuccess || hipDeviceSynchronize() != hipSuccess) {
            (void)hipGetLastError();
            continue;
        }
        std::vector<Block> blocks;
        {
            std::lock_guard<std::mutex> table(g_mu);
            blocks = p->take_blocks(uses);
            if (p->empty() && !p->retired) {
                p->retired = true;
                auto& list = p->owner.recording ? g_graphs : g_streams;
                for (size_t i = 0; i < list.size(); ++i)
                    if (list[i] == p) { list.erase(list.begin() + (long)i); break; }
            }
        }
        p->free_blocks(blocks);
    }
    (void)hipSetDevice(current);
    (void)hipGetLastError();
}
