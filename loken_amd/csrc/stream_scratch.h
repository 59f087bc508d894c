// Scratch memory of the launchers that need some between their kernels: one grow-only buffer per
// (device, stream, use), freed by loken_stream_scratch_release (moe_decode.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>

// A buffer per use, so that a launcher may call another one between filling and reading its own.
enum LkScratchUse { LK_SCRATCH_LAUNCHER = 0, LK_SCRATCH_BLOCK = 1, LK_SCRATCH_ROUTER = 2 };

// Held from a reservation until the launches that use the buffer are on the stream: the buffer belongs to
// the stream, and another thread's launches landing between a launcher's kernels would overwrite it.
// Recursive: a launcher that holds it calls others.
std::recursive_mutex& lk_scratch_mutex();

// `bytes` of the stream's buffer for `use`, 256-byte aligned, not initialised; null when there is no memory
// or when the buffer would have to grow while `stream` records a graph. Caller holds lk_scratch_mutex().
void* lk_reserve_scratch(size_t bytes, hipStream_t stream, LkScratchUse use);
