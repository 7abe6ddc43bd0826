// Host side of the device layer: the pool of idle device blocks and streams,
// and the wait for a kernel's report.
// No kernels and no header of theirs, so it compiles with any C++ compiler
// and its rules are tested without a GPU (tests/test_pool.py).
#pragma once

#include <hip/hip_runtime_api.h>
#include <stddef.h>
#include <stdint.h>

#include <vector>

// Reads the bounds of this process's device memory from the environment, once
// per handle: PARRSB_AMD_POOL_MB (idle blocks per device, default 4096; 0:
// keep nothing) and PARRSB_AMD_MEM_LIMIT_MB (all blocks; unset: no limit).
void rsb_pool_settings(void);
// A block of device memory, from the pool where one fits, else hipMalloc.
hipError_t rsb_pool_malloc(void **p, size_t bytes);
// Back to the device now (hipFree waits for it).
hipError_t rsb_pool_free(const void *p);
// To the pool: only a block that no queued work uses any more.
void rsb_pool_release(const void *p);

// The stream, events and pinned ring of closed handles, likewise.
struct rsb_stream_set {
  hipStream_t stream;
  hipEvent_t ev[4];
  int *ring;  // pinned: the counts a solve's kernels report to the host
};
bool rsb_pool_take_streams(int device, rsb_stream_set *out);
bool rsb_pool_give_streams(int device, const rsb_stream_set &in);
void rsb_destroy_streams(const rsb_stream_set &s);
// One more handle of the device has closed.
void rsb_pool_tick(int device);

// The library's allocator (noalloc.hip): rsb_pool_malloc and its counterparts,
// or the fixed array inside an allocation-free call.
hipError_t rsb_dev_malloc(void **p, size_t bytes);
hipError_t rsb_dev_free(const void *p);
void rsb_dev_release(const void *p);
// Gives back the blocks that a stream's work has used: released once the
// stream has drained; freed if it cannot be shown to have, since a block of
// the pool may go to any thread and stream.  Returns whether it has.
bool rsb_drain_release(hipStream_t st, const std::vector<const void *> &blocks);

// The schedule flags (hipDeviceSchedule*) of the current device.
unsigned rsb_schedule(void);
// Waits until a kernel on the stream has set *flag (pinned memory), as the
// schedule flags ask: looking all the time (Auto, Spin), with the rest of the
// time slice given away after each look (Yield), or asleep in the runtime
// until the stream has drained (BlockingSync).  hipErrorNotReady: the stream
// has ended without setting it.
hipError_t rsb_await(hipStream_t st, const int *flag, unsigned schedule);
