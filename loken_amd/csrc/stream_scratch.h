// Scratch memory of the launchers that need some between their kernels: per (device, stream) a few grow-only
// buffers, one per use. Stream order keeps the launches of one stream apart, so nothing waits on events: a
// hipEventRecord after every launch, which one shared buffer per device would need, costs the queue 4 us each
// (measured: launches back to back 2.4 us apart, with a record after each 6.4).
//
// A recorded graph replays on whatever stream its program picks, beside calls and graphs that stream order does
// not keep apart from it. So what is recorded gets buffers of its own, per (capture, stream), that no call and no
// other graph uses, and keeps them until the release.
//
// Past LK_SCRATCH_STREAMS streams of a device (destroyed ones count until the release) the further ones share one
// set of buffers, ordered by such events.
#pragma once

#include <hip/hip_runtime.h>

#include <memory>
#include <mutex>

// A buffer per use, so that a launcher may call another one between filling and reading its own.
enum LkScratchUse {
    LK_SCRATCH_LAUNCHER,   // expert launchers: quantized rows, pair rows
    LK_SCRATCH_BLOCK,      // expert block: what passes between its launches
    LK_SCRATCH_ROUTER,     // gate logits
    LK_SCRATCH_LINEAR,     // host linear: quantized rows
    LK_SCRATCH_FIXUP,      // tiled matmul: partial products of a cut K
    LK_SCRATCH_TOKENS,     // f16 tiles: token operands
    LK_SCRATCH_USES
};

struct LkScratchPool;

// The scratch of `stream` on the current device (hipStreamPerThread: the calling thread's), held from before a
// reservation until the launches that use the buffer are on the stream: another thread's launches on the same
// stream, landing between a launcher's kernels, would overwrite it. A launcher that holds it may call others.
class LkScratch {
  public:
    explicit LkScratch(hipStream_t stream);
    ~LkScratch();
    LkScratch(const LkScratch&) = delete;
    LkScratch& operator=(const LkScratch&) = delete;

    // `bytes` for `use`, 256-byte aligned, not initialised; null when there is no memory. While the stream records a
    // graph, also null where no call of the device outside a capture has needed that much (the program warms up
    // before it records, on any stream), and past LK_SCRATCH_GRAPH_BYTES. A buffer grows by a quarter more than asked;
    // the one it replaces is freed first, which waits for the device (so a launcher queues what reads a buffer before it
    // asks for more of the same use), or kept until the release where a graph's nodes hold its address.
    void* get(LkScratchUse use, size_t bytes);

    // A number below LK_SCRATCH_TICKETS that no other stream's scratch has: which of an array of counters in device memory a kernel
    // may count its workgroups in. A launch finds its counter at zero and leaves it there. -1 where all are taken, and while the stream
    // records a graph.
    int ticket() const;

    // Whether the stream records a graph, which keeps what it takes.
    bool recording() const;

  private:
    hipStream_t stream_;
    std::shared_ptr<LkScratchPool> pool_;
    std::unique_lock<std::recursive_mutex> lock_;
};

// Streams of a device with buffers of their own.
constexpr int LK_SCRATCH_STREAMS = 32;
// Streams' scratches with a counter of their own.
constexpr int LK_SCRATCH_TICKETS = 4096;
// What all recorded graphs of a device may hold together.
constexpr size_t LK_SCRATCH_GRAPH_BYTES = (size_t)32 << 30;
// The uses of the host linears, and those of everything else: each side gives back its own.
constexpr unsigned LK_SCRATCH_OF_LINEARS = 1u << LK_SCRATCH_LINEAR | 1u << LK_SCRATCH_FIXUP;
constexpr unsigned LK_SCRATCH_OF_LAUNCHERS = (1u << LK_SCRATCH_USES) - 1 - LK_SCRATCH_OF_LINEARS;
// Gives back what the streams and graphs of `device` (-1: of every device) hold for `uses`, a bit per use. Waits for
// the device; a graph recorded over any of it must not be replayed after.
void lk_stream_scratch_release(int device, unsigned uses);
