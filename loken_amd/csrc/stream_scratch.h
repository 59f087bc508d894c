// Scratch memory of the launchers that need some between their kernels: per (device, stream) a few grow-only
// buffers, one per use. Stream order keeps the launches of one stream apart, so nothing waits on events: a
// hipEventRecord after every launch, which one shared buffer per device would need, costs the queue 4 us each
// (measured: launches back to back 2.4 us apart, with a record after each 6.4).
#pragma once

#include <hip/hip_runtime.h>

#include <memory>
#include <mutex>
#include <vector>

// A buffer per use, so that a launcher may call another one between filling and reading its own.
enum LkScratchUse {
    LK_SCRATCH_LAUNCHER,   // expert launchers: quantized rows, pair rows
    LK_SCRATCH_BLOCK,      // expert block: what passes between its launches
    LK_SCRATCH_ROUTER,     // gate logits
    LK_SCRATCH_LINEAR,     // host linear: quantized rows
    LK_SCRATCH_FIXUP,      // tiled matmul: partial products of a cut K
    LK_SCRATCH_TOKENS,     // wide tiles: token operands
    LK_SCRATCH_USES
};

class LkStreamScratch {
  public:
    explicit LkStreamScratch(int device) : device_(device) {}
    LkStreamScratch(const LkStreamScratch&) = delete;
    LkStreamScratch& operator=(const LkStreamScratch&) = delete;

    // Held from a reservation until the launches that use the buffer are on the stream: another thread's launches
    // on the same stream, landing between a launcher's kernels, would overwrite it. Recursive: a launcher that
    // holds it calls others.
    std::recursive_mutex mu;
    // `bytes` for `use`, 256-byte aligned, not initialised; null when there is no memory. Caller holds mu. A stream
    // that records a graph allocates nothing: what its own buffer does not hold it takes from another stream's of
    // the device (a program warms up on one stream and records on another; the graph's replays are then the
    // program's to keep apart from that stream's calls), null when none is large enough. Outgrown buffers stay
    // (queued kernels and recorded graphs may still use them) until the release; a buffer grows by a quarter more
    // than asked, so they add up to a few times the largest.
    void* get(LkScratchUse use, size_t bytes, hipStream_t stream);
    void free_all();   // caller holds mu and knows that nothing queued uses the buffers

    int device() const { return device_; }
    bool recorded = false;   // a graph recorded on this stream may hold the buffers' addresses: not given up for another's
    unsigned long long used_at = 0;

  private:
    struct Block;
    int device_;
    std::shared_ptr<Block> now_[LK_SCRATCH_USES];
    std::vector<std::shared_ptr<Block>> kept_;
    static std::vector<std::weak_ptr<Block>>& blocks();   // of every stream, under the table's lock
};

// The current device's scratch for `stream` (hipStreamPerThread: the calling thread's). At most LK_SCRATCH_STREAMS
// streams of a device hold some without having recorded a graph: past that the least recently used one gives its up.
constexpr int LK_SCRATCH_STREAMS = 32;
std::shared_ptr<LkStreamScratch> lk_stream_scratch(hipStream_t stream);
// Gives back what the streams of `device` hold (-1: of every device). Waits for the device.
void lk_stream_scratch_release(int device);
