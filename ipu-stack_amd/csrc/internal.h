// Internal host-side declarations shared by the libipus translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "../../include/ipus.h"

#include <atomic>
#include <mutex>
#include <unordered_map>

struct ipus_context {
  int device = 0;
  hipStream_t stream = nullptr;
  // Buffers allocated through this context and not yet freed (pointer ->
  // bytes); ipus_context_destroy releases whatever is left.
  std::mutex live_mutex;
  std::unordered_map<void*, size_t> live;
  // Failure injection (ipus_context_inject_launch_failure): after
  // inject_after more launches, the next one returns inject_status.
  uint32_t inject_after = 0;
  int inject_status = 0;
  // Workspace of the kernels that split a reduction over workgroups
  // (context_workspace): allocated with the context, not counted among the
  // buffers above.
  void* workspace = nullptr;
  uint32_t* workspace_counters = nullptr;
  // ipus_session_capture is recording this context's stream into a graph
  // that will only be launched on it.
  std::atomic<bool> capturing_session{false};
};

namespace ipus {

struct Workspace;
// The context's workspace, for a launch on its stream: launches there run one
// after the other, whichever threads enqueue them, so they can share it.
// Empty where the allocation failed, and while a caller records the stream
// into a graph of its own (which it may launch on other streams, several at
// once): the unsplit kernels run then.
Workspace context_workspace(const ipus_context* ctx);
// The context's stream is being recorded into a graph (or cannot tell).
bool stream_recorded(const ipus_context* ctx);

// Records a formatted message as the thread's last error and returns `code`.
int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
int hip_fail(hipError_t e, const char* what);
// Makes the context's device current for the calling thread.
int use_device(const ipus_context* ctx);
// Turns a launcher status into a recorded error for `symbol`.
int check_launch(int status, const char* symbol);

int run_flat_add(ipus_context* c, void* o, const void* const* i, const uint32_t* s, int precision);
int run_broadcast_add(ipus_context* c, void* o, const void* const* i, const uint32_t* s,
                      int precision);

}  // namespace ipus
