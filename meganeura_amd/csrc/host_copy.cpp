// Copies between ordinary host memory and the device, through pinned memory of the context's own.
//
// The runtime's copy of pageable memory stages or pins page by page and waits in between: a 196 KB read takes
// 83 us, 1.36 MB 65 us up and 85 us down, 64 MB up 2210 us, where the same copies of pinned memory take
// 11, 31, 32 and 1200 us.  The CPU moves cached data at some 85 GB/s (1.36 MB 16 us) and data from
// DRAM at 29 GB/s per thread, so:
//   up to kSmall: through a ring that is handed out front to back, in chunks, so that the CPU fills the
//     next chunk while the last one travels; writes need not be waited for (the stream keeps them in
//     order with the launches that read them); launches, not copy engine commands, move the chunks
//     (copy_bytes_kernel), except reads on an idle stream;
//   beyond (uploads from kLargeIn on): the ring as slots of kSlot, up to kWorkers threads with two slots
//     each that take the chunks in turn (one thread's 29 GB/s is half of what the bus takes: 64 MB 2650 us with one thread, 1590
//     with four).  The threads live as long as the call.
// Measured, before -> after: the eight-layer decode step of a session 147 -> 124 us, two layers of 333
// rows 460 -> 410 us, a 4096 x 4096 weight from f32 and its packed bytes back 3400 -> 2470 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <thread>

#include "mgn_internal.h"

namespace mgn {
namespace {

constexpr size_t kSlot = (size_t)2 << 20, kSlots = 8, kRing = kSlot * kSlots;
constexpr int kWorkers = (int)kSlots / 2;
constexpr size_t kSmall = (size_t)4 << 20;
// Uploads between these two go the runtime's way, which pins the pages: one thread fills the ring at what DRAM
// gives it, and four cost their start.  Whole upload or weight from f32, ring or slots : runtime, us: 2 MB 108 : 98,
// 3.5 MB weight 285 : 236, 8 MB weight 460 : 415, 12 MB 410 : 352 from the caches, 438 : 419 from memory,
// 16 MB 510 : 460 and 531 : 582, 32 MB 863 : 920 and 876 : 1139.
constexpr size_t kSmallIn = (size_t)2 << 20, kLargeIn = (size_t)16 << 20;
constexpr size_t kChunk = (size_t)1 << 20, kChunkOut = (size_t)512 << 10;
constexpr size_t kEvents = sizeof(HostStage::done) / sizeof(ihipEvent_t*);
static_assert(kSmallIn <= kSmall && kSmall / kChunkOut <= kEvents && kSlots <= kEvents, "an event per chunk, and per slot");

// The context's device while it lives, the caller's afterwards: events belong to the device that is current when they
// are made, and record on no other device's stream.
class OnDevice {
 public:
  explicit OnDevice(int device) : mine_(device) {
    if (hipGetDevice(&before_) != hipSuccess) before_ = mine_;
    if (before_ != mine_) (void)hipSetDevice(mine_);
  }
  ~OnDevice() {
    if (before_ != mine_) (void)hipSetDevice(before_);
  }
  OnDevice(const OnDevice&) = delete;
  OnDevice& operator=(const OnDevice&) = delete;

 private:
  int mine_, before_ = 0;
};

// The context's ring and events (its device is current); false: there is no pinned memory to be had.
bool have_stage(mgn_ctx* ctx) {
  HostStage& st = ctx->stage;
  if (st.ring) return true;
  if (st.refused) return false;
  hipError_t e = hipHostMalloc((void**)&st.ring, kRing, hipHostMallocDefault);
  if (e == hipSuccess) e = hipHostGetDevicePointer((void**)&st.ring_dev, st.ring, 0);
  for (size_t i = 0; e == hipSuccess && i < kEvents; i++) e = hipEventCreateWithFlags(&st.done[i], hipEventDisableTiming);
  if (e == hipSuccess) return true;
  (void)hipGetLastError();
  release_host_stage(ctx);
  st.refused = true;
  return false;
}

// Memory the runtime knows (pinned, managed, a device's) is copied by the runtime as it is.
bool pageable(const void* p) {
  hipPointerAttribute_t at{};
  if (hipPointerGetAttributes(&at, p) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return at.type == hipMemoryTypeUnregistered;
}

// `bytes` between the ring (from `ring_off` on) and the device, queued on the stream.
hipError_t queue_copy(mgn_ctx* ctx, char* dev, size_t ring_off, size_t bytes, bool in) {
  if (((uintptr_t)dev & 15) == 0)
    return (hipError_t)(in ? launch_copy_bytes(ctx->stream, dev, ctx->stage.ring_dev + ring_off, bytes)
                           : launch_copy_bytes(ctx->stream, ctx->stage.ring_dev + ring_off, dev, bytes));
  char* const host = ctx->stage.ring + ring_off;
  return in ? hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, ctx->stream)
            : hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, ctx->stream);
}

// More than kSmall bytes; the stream is idle on return.
hipError_t copy_large(mgn_ctx* ctx, char* dev, char* host, size_t bytes, bool in) {
  hipError_t e = hipStreamSynchronize(ctx->stream);  // (the ring is free)
  if (e != hipSuccess) return e;
  ctx->stage.used = 0;
  const size_t chunks = (bytes + kSlot - 1) / kSlot;
  std::atomic<size_t> next{0};
  std::atomic<int> error{(int)hipSuccess};
  auto work = [&](int worker) {
    hipError_t err = worker ? hipSetDevice(ctx->device) : hipSuccess;  // (a thread starts on device 0)
    size_t busy[2] = {0, 0};  // chunk + 1 that travels through the slot
    auto size_of = [&](size_t c) { return std::min(kSlot, bytes - c * kSlot); };
    // waits for what travels through slot s; on the way out, takes it from there
    auto finish = [&](int s) {
      if (!busy[s]) return;
      const size_t c = busy[s] - 1;
      const hipError_t we = hipEventSynchronize(ctx->stage.done[worker * 2 + s]);
      if (err == hipSuccess) err = we;
      if (!in && err == hipSuccess) std::memcpy(host + c * kSlot, ctx->stage.ring + (worker * 2 + s) * kSlot, size_of(c));
      busy[s] = 0;
    };
    int s = 0;
    for (; err == hipSuccess && error.load(std::memory_order_relaxed) == (int)hipSuccess; s ^= 1) {
      const size_t c = next.fetch_add(1);
      if (c >= chunks) break;
      finish(s);
      if (err != hipSuccess) break;
      const size_t slot = (worker * 2 + s) * kSlot;
      if (in) std::memcpy(ctx->stage.ring + slot, host + c * kSlot, size_of(c));
      err = queue_copy(ctx, dev + c * kSlot, slot, size_of(c), in);
      if (err == hipSuccess) err = hipEventRecord(ctx->stage.done[worker * 2 + s], ctx->stream);
      if (err == hipSuccess) busy[s] = c + 1;
    }
    finish(s);
    finish(s ^ 1);
    if (err != hipSuccess) error.store((int)err);
  };
  const unsigned cpus = std::thread::hardware_concurrency();
  const int wanted = (int)std::min<size_t>({(size_t)kWorkers, (chunks + 1) / 2, cpus ? cpus : 1});
  std::thread helpers[kWorkers - 1];
  for (int i = 1; i < wanted; i++) {
    try {
      helpers[i - 1] = std::thread(work, i);
    } catch (const std::exception&) {
      break;  // no more threads, or no memory for one: those there are take all chunks
    }
  }
  work(0);
  for (std::thread& t : helpers)
    if (t.joinable()) t.join();
  e = hipStreamSynchronize(ctx->stream);
  return error.load() != (int)hipSuccess ? (hipError_t)error.load() : e;
}

// A piece of the ring for `bytes` (at most kSmall).
hipError_t ring_piece(mgn_ctx* ctx, size_t bytes, size_t* out) {
  HostStage& st = ctx->stage;
  const size_t need = (bytes + 255) & ~(size_t)255;
  if (st.used + need > kRing) {
    if (const hipError_t e = hipStreamSynchronize(ctx->stream)) return e;
    st.used = 0;
  }
  *out = st.used;
  st.used += need;
  return hipSuccess;
}

}  // namespace

int copy_in(mgn_ctx* ctx, void* dev, const void* host, size_t bytes) {
  if (bytes == 0) return 0;
  const OnDevice on(ctx->device);
  if ((bytes > kSmallIn && bytes < kLargeIn) || !pageable(host) || !have_stage(ctx)) {
    hipError_t e = hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    return (int)e;
  }
  if (bytes > kSmallIn) return (int)copy_large(ctx, (char*)dev, (char*)const_cast<void*>(host), bytes, true);
  size_t piece;
  if (const hipError_t e = ring_piece(ctx, bytes, &piece)) return (int)e;
  for (size_t o = 0; o < bytes; o += kChunk) {
    const size_t b = std::min(kChunk, bytes - o);
    std::memcpy(ctx->stage.ring + piece + o, (const char*)host + o, b);
    if (const hipError_t e = queue_copy(ctx, (char*)dev + o, piece + o, b, true)) return (int)e;
  }
  return 0;
}

int copy_out(mgn_ctx* ctx, void* host, const void* dev, size_t bytes) {
  if (bytes == 0) return (int)hipStreamSynchronize(ctx->stream);
  const OnDevice on(ctx->device);
  if (!pageable(host) || !have_stage(ctx)) {
    hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    return (int)e;
  }
  if (bytes > kSmall) return (int)copy_large(ctx, (char*)const_cast<void*>(dev), (char*)host, bytes, false);
  size_t piece;
  if (const hipError_t e = ring_piece(ctx, bytes, &piece)) return (int)e;
  char* const ring = ctx->stage.ring + piece;
  const char* const src = (const char*)dev;
  // behind a kernel a launch is the faster one (196 KB and the wait 17 against 25 us), on an idle stream
  // the copy engine (11.3 against 14.8)
  const bool idle = hipStreamQuery(ctx->stream) == hipSuccess;
  if (!idle) (void)hipGetLastError();
  const size_t chunks = (bytes + kChunkOut - 1) / kChunkOut;
  for (size_t c = 0; c < chunks; c++) {
    const size_t o = c * kChunkOut, b = std::min(kChunkOut, bytes - o);
    hipError_t e = idle ? hipMemcpyAsync(ring + o, src + o, b, hipMemcpyDeviceToHost, ctx->stream)
                        : queue_copy(ctx, const_cast<char*>(src) + o, piece + o, b, false);
    if (e == hipSuccess && c + 1 < chunks) e = hipEventRecord(ctx->stage.done[c], ctx->stream);
    if (e != hipSuccess) return (int)e;
  }
  for (size_t c = 0; c < chunks; c++) {
    const size_t o = c * kChunkOut, b = std::min(kChunkOut, bytes - o);
    if (const hipError_t e = c + 1 < chunks ? hipEventSynchronize(ctx->stage.done[c]) : hipStreamSynchronize(ctx->stream)) return (int)e;
    std::memcpy((char*)host + o, ring + o, b);
  }
  ctx->stage.used = 0;
  return 0;
}

void release_host_stage(mgn_ctx* ctx) {
  HostStage& st = ctx->stage;
  for (ihipEvent_t*& e : st.done) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  if (st.ring) (void)hipHostFree(st.ring);
  st.ring = nullptr;
  st.used = 0;
}

}  // namespace mgn
