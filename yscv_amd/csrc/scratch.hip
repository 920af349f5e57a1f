// Scratch memory of calls that bring none of their own (prepared activations, partial sums, quantised copies).
//
// A hipMallocAsync / hipFreeAsync pair costs 15 us of host time on this runtime, as much as the kernels of a small call
// together (24 bf16 rows x 256 x 512: 26.5 us a call against 11.7 with the caller's own workspace), so blocks are kept.  On
// the default stream a block costs nothing measurable (7.9 us a call, 8.2 with the caller's workspace), on another stream 4 us
// (12.1): the capture query, the wait for the last use, the event behind this one.
// There is one block for the default stream and eight for other streams (least recently used one first when
// a ninth stream comes).  A block is used by one call at a time: its lock is held from the first launch that uses it to
// the last, so two threads on one stream cannot interleave their launches, and the stream runs them in that order.
// The default stream cannot be destroyed, so reuse there needs nothing more.  Any other handle may have been destroyed
// and reissued between two calls, so the end of every use is recorded as an event and the next use waits for it.
// Bounded: a block keeps at most kKeep bytes (576 MiB of 288 GB in all); larger requests, and requests of a stream that
// is being captured into a graph (whose memory must belong to the graph), go to the stream-ordered allocator as before.
// yscv_hip_shutdown gives the blocks back.
#include "common.hpp"

namespace yscv {

namespace {

constexpr size_t kKeep = (size_t)64 << 20;
constexpr size_t kFirst = (size_t)1 << 20;  // smallest block: most calls of most programs fit, few regrow
constexpr int kSlots = 9;                   // 0: default stream

}  // namespace

struct ScratchSlot {
  std::mutex busy;
  void *p = nullptr;
  size_t cap = 0;
  int device = -1;
  hipStream_t owner = nullptr;  // guarded by g_pick, like `taken` and `used`
  bool taken = false;
  uint64_t used = 0;
  hipEvent_t end = nullptr;  // end of the last use (slots of other streams)
};

static ScratchSlot g_slots[kSlots];
static std::mutex g_pick;
static uint64_t g_tick = 0;

static ScratchSlot *pick_slot(hipStream_t s) {
  if (s == nullptr) return &g_slots[0];
  std::lock_guard<std::mutex> lock(g_pick);
  ScratchSlot *best = nullptr;
  for (int i = 1; i < kSlots; i++) {
    ScratchSlot &c = g_slots[i];
    if (c.taken && c.owner == s) {
      best = &c;
      break;
    }
    if (!best || (best->taken && (!c.taken || c.used < best->used))) best = &c;
  }
  best->taken = true;
  best->owner = s;
  best->used = ++g_tick;
  return best;
}

static int32_t alloc_failed(hipError_t e, size_t bytes) {
  return set_error(e == hipErrorOutOfMemory ? YSCV_HIP_ERR_OOM : YSCV_HIP_ERR_DEVICE, "scratch allocation of %zu bytes failed: %s",
                   bytes, hipGetErrorString(e));
}

bool stream_capturing(hipStream_t s) {
  if (s == nullptr) return false;
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(s, &st) != hipSuccess || st != hipStreamCaptureStatusNone;
}

int32_t Scratch::take(size_t bytes, hipStream_t stream) {
  s = stream;
  if (bytes == 0) bytes = 4;
  if (bytes > kKeep || stream_capturing(stream)) {
    const hipError_t e = hipMallocAsync(&p, bytes, stream);
    if (e != hipSuccess) {
      p = nullptr;
      return alloc_failed(e, bytes);
    }
    return YSCV_HIP_OK;
  }
  slot = pick_slot(stream);
  slot->busy.lock();
  int device = 0;
  hipError_t e = hipGetDevice(&device);
  // (an event belongs to one device: another one's is drained on the host and dropped with the block.  The event is not
  // asked whether it has passed: such a query ends the capture that another stream may be under.)
  if (e == hipSuccess && slot->end && slot->device == device) e = hipStreamWaitEvent(stream, slot->end, 0);
  if (e == hipSuccess && slot->p && (slot->device != device || slot->cap < bytes)) {
    if (slot->device == device) {
      e = hipFreeAsync(slot->p, stream);  // behind the wait above, so behind its last use
    } else {
      (void)hipSetDevice(slot->device);
      e = hipFree(slot->p);  // waits for that device
      if (slot->end) (void)hipEventDestroy(slot->end);
      slot->end = nullptr;
      (void)hipSetDevice(device);
    }
    slot->p = nullptr;
    slot->cap = 0;
  }
  if (e == hipSuccess && !slot->p) {
    size_t cap = kFirst;
    while (cap < bytes) cap *= 2;
    e = hipMallocAsync(&slot->p, cap, stream);
    slot->cap = e == hipSuccess ? cap : 0;
    slot->device = device;
    if (e != hipSuccess) slot->p = nullptr;
  }
  if (e == hipSuccess && stream != nullptr && !slot->end) e = hipEventCreateWithFlags(&slot->end, hipEventDisableTiming);
  if (e != hipSuccess) {
    slot->busy.unlock();
    slot = nullptr;
    return alloc_failed(e, bytes);
  }
  p = slot->p;
  return YSCV_HIP_OK;
}

Scratch::~Scratch() {
  if (slot) {
    if (slot->end && hipEventRecord(slot->end, s) != hipSuccess) (void)hipStreamSynchronize(s);
    slot->busy.unlock();
  } else if (p) {
    (void)hipFreeAsync(p, s);
  }
}

void release_scratch() {
  for (ScratchSlot &c : g_slots) {
    std::lock_guard<std::mutex> busy(c.busy);
    if (c.p) {
      int device = 0;
      (void)hipGetDevice(&device);
      (void)hipSetDevice(c.device);
      (void)hipFree(c.p);
      if (c.end) (void)hipEventDestroy(c.end);
      (void)hipSetDevice(device);
    }
    c.p = nullptr;
    c.end = nullptr;
    c.cap = 0;
    std::lock_guard<std::mutex> pick(g_pick);
    c.taken = false;
    c.owner = nullptr;
  }
}

}  // namespace yscv
