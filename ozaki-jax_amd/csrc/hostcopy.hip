// Copies between pageable host memory and the device through pinned memory.
// Host threads move pieces while others are on the link, so the transfer, the
// host copies and the page faults of a fresh output array overlap each other
// and the kernels queued before the copy.
//
// What bounds them: the link (55 GB/s down).  Down, one kernel writes the
// pinned memory and reports each piece as it lands: queued copies of 4 MiB with
// an event each left about 15 us between them (32 MiB: 0.80 ms into a warm array,
// 1.31 as one copy and a host copy behind it; the link alone takes 0.61).  Up,
// the host threads come first, so their pieces go as copies of a slot; large
// transfers go so both ways, in larger slots, since queued copies also run
// beside a kernel that holds every CU (a product in row halves).
//
// Pinned memory serves one copy at a time, and no caller waits for what another
// has queued on its stream.  Copies through slots take turns, each once its
// stream has drained: queued behind kernels they would keep the slots, and the
// DMA engine they are queued on, from everyone.  (The second of two uploads in a
// row goes behind the first all the same: a product of 400^3 NumPy arrays takes
// 230 to 255 us, 265 where it waits, 225 where neither does.)  The small copy
// down, a kernel, does not wait either, which would cost it about 40 us (56 -> 95
// at 1 MiB, 235 -> 330 at 8): it holds the memory from its launch on, and a
// caller that finds it held takes the runtime's own copy.
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <string.h>
#include <thread>
#include <vector>

#include "common.h"

namespace ozk {

constexpr size_t kPiece = 512 << 10;
constexpr uintptr_t kHugePage = 2 << 20;

// Held while a copy uses the pinned memory at `staging`, of copy_out or of
// copy_slots.  (Other memory of the same kind may share the mutex; of the other
// kind not, since copy_out holds it while its stream is busy.)
static std::mutex& staging_turn(const void* staging, bool slots) {
  static std::mutex turns[2][64];
  return turns[slots][((uintptr_t)staging >> 20) % 64];
}

// Waits for the stream.  A stream that the runtime knows to be idle is asked
// (0.3 us; synchronising it can take 60); one whose last work is a copy_out is
// not known to be, and asking would cost 15 us on top of the 16 of the wait.
// g_copied_out, the stream of the last copy_out, only chooses between the two.
static const hipStream_t kNoStream = (hipStream_t)(intptr_t)-1;
static std::atomic<hipStream_t> g_copied_out{kNoStream};
static hipError_t drain(hipStream_t st) {
  const bool ask = g_copied_out.exchange(kNoStream, std::memory_order_relaxed) != st;
  return ask && hipStreamQuery(st) == hipSuccess ? hipSuccess : hipStreamSynchronize(st);
}

// ---------------------------------------------------------------- down
constexpr int kOutThreads = 256, kOutUnits = 4;
constexpr size_t kOutBytes = (size_t)kOutThreads * kOutUnits * 16;  // 16 KiB a workgroup
constexpr int kOutPerPiece = (int)(kPiece / kOutBytes);

constexpr int kOutGrid = 128;

constexpr int kAwakePolls = 8192;  // about 0.3 ms

// src -> dst (pinned host memory, 16-byte aligned) in blocks of 16 KiB,
// dealt to the workgroups in order: kOutGrid of them fill the link and few
// enough are under way at once for the pieces to land one after the other
// (one workgroup per block had every piece under way, and none land early:
// 0.95 ms for 32 MiB).  The last workgroup of a piece to finish stores `seq` to
// its flag (host memory) and leaves its counter at zero.  V: the widest type
// src allows.
template <typename V>
__global__ __launch_bounds__(kOutThreads) void copy_out_kernel(const char* __restrict__ src,
                                                               char* __restrict__ dst,
                                                               size_t bytes, int blocks,
                                                               uint32_t* __restrict__ count,
                                                               uint32_t* __restrict__ flags,
                                                               uint32_t seq) {
  constexpr int kPer = (int)(kOutBytes / sizeof(V)) / kOutThreads;
  constexpr int kBatch = kPer < 8 ? kPer : 8;  // loads in flight together
  for (int blk = blockIdx.x; blk < blocks; blk += gridDim.x) {
    const size_t b0 = (size_t)blk * kOutBytes;
    const size_t n = bytes - b0 < kOutBytes ? bytes - b0 : kOutBytes;
    const size_t whole = n / sizeof(V);
    const V* const s = (const V*)(src + b0);
    V* const d = (V*)(dst + b0);
    for (int i0 = 0; i0 < kPer; i0 += kBatch) {
      V v[kBatch];
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        const size_t k = (size_t)(i0 + i) * kOutThreads + threadIdx.x;
        if (k < whole) v[i] = s[k];
      }
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        const size_t k = (size_t)(i0 + i) * kOutThreads + threadIdx.x;
        if (k < whole) d[k] = v[i];
      }
    }
    for (size_t k = whole * sizeof(V) + threadIdx.x; k < n; k += kOutThreads)
      dst[b0 + k] = src[b0 + k];
    __threadfence_system();  // this thread's bytes are in host memory
    __syncthreads();
    if (threadIdx.x == 0) {
      const int piece = blk / kOutPerPiece, left = blocks - piece * kOutPerPiece;
      const uint32_t of = (uint32_t)(left < kOutPerPiece ? left : kOutPerPiece);
      if (__hip_atomic_fetch_add(count + piece, 1u, __ATOMIC_ACQ_REL,
                                 __HIP_MEMORY_SCOPE_AGENT) == of - 1) {
        __hip_atomic_store(count + piece, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(flags + piece, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
  }
}

static std::atomic<uint32_t> g_out_seq{0};

struct OutJob {
  char* host;
  const char* dev;
  size_t bytes, batch;  // batch: bytes a launch copies
  char* staging;
  uint32_t *count, *flags;
  size_t half;  // bytes between the staging of even and odd batches
  hipStream_t st;
  int device;
  std::vector<std::atomic<uint32_t>> seq;  // per batch: 0 until launched
  std::vector<std::atomic<int>> left;      // pieces of a batch still to be taken
  std::atomic<size_t> touch{0}, touched{0};  // the output's huge pages taken, written
  std::atomic<size_t> next{0};                // next piece
  std::atomic<int> err{0};
  std::atomic<bool> lost{false};
  std::mutex gate;
  std::condition_variable gate_cv;
  std::atomic<bool> open{false};  // the first piece is there (or something failed)

  explicit OutJob(size_t batches) : seq(batches), left(batches) {}
  size_t batches() const { return seq.size(); }
  size_t batch_bytes(size_t b) const { return b + 1 < batches() ? batch : bytes - b * batch; }
  bool failed() const { return err.load(std::memory_order_relaxed) || lost.load(); }
  bool ok(hipError_t e) {
    if (e == hipSuccess) return true;
    int none = 0;
    err.compare_exchange_strong(none, (int)e);
    return false;
  }
  void launch(size_t b) {
    uint32_t q = g_out_seq.fetch_add(1) + 1;
    while (q == 0) q = g_out_seq.fetch_add(1) + 1;
    const char* const s = dev + b * batch;
    char* const d = staging + (b & 1) * half;
    uint32_t* const c = count + (b & 1) * (half / kPiece);
    uint32_t* const f = flags + (b & 1) * (half / kPiece);
    const size_t n = batch_bytes(b);
    const int blocks = (int)((n + kOutBytes - 1) / kOutBytes);
    const dim3 grid((unsigned)(blocks < kOutGrid ? blocks : kOutGrid));
#define OZK_OUT(V)                                                                            \
  hipLaunchKernelGGL(copy_out_kernel<V>, grid, dim3(kOutThreads), 0, st, s, d, n, blocks, c, f, q)
    if ((uintptr_t)s % 16 == 0) OZK_OUT(uint4);
    else if ((uintptr_t)s % 8 == 0) OZK_OUT(uint64_t);
    else OZK_OUT(uint8_t);
#undef OZK_OUT
    ok(hipGetLastError());
    seq[b].store(q, std::memory_order_release);
  }
  // Waits for piece k of batch b; false when something failed.  The stream
  // is asked for its state now and then: an error, or a drained stream whose
  // piece never came, ends the wait.
  bool wait(size_t b, size_t k) {
    uint32_t q;
    while ((q = seq[b].load(std::memory_order_acquire)) == 0) {
      if (failed()) return false;
      std::this_thread::yield();
    }
    const uint32_t* const f = flags + (b & 1) * (half / kPiece) + k;
    for (;;) {
      for (int i = 0; i < 4096; ++i) {
        if (__atomic_load_n(f, __ATOMIC_ACQUIRE) == q) return true;
        __builtin_ia32_pause();
      }
      if (failed()) return false;
      const hipError_t e = hipStreamQuery(st);
      if (e == hipErrorNotReady) continue;
      if (!ok(e)) return false;
      if (__atomic_load_n(f, __ATOMIC_ACQUIRE) == q) return true;
      lost.store(true);
      return false;
    }
  }
  // Lets the other threads at the pieces.
  void begin() {
    {
      std::lock_guard<std::mutex> g(gate);
      open.store(true, std::memory_order_release);
    }
    gate_cv.notify_all();
  }
  void work(bool caller) {
    // the output's pages, while the device is still busy before the copy; a
    // huge page by one thread (several that fault one each zero a page for it)
    const uintptr_t h0 = (uintptr_t)host, base = h0 & ~(kHugePage - 1);
    const size_t pages = (h0 + bytes - base + kHugePage - 1) / kHugePage;
    for (size_t p; (p = touch.fetch_add(1)) < pages; touched.fetch_add(1)) {
      const uintptr_t a = base + p * kHugePage;
      for (uintptr_t o = a < h0 ? h0 : a; o < a + kHugePage && o < h0 + bytes;
           o = (o & ~(uintptr_t)4095) + 4096)
        *(volatile char*)o = 0;
    }
    // no piece may land on a page that another thread still writes
    while (touched.load(std::memory_order_acquire) < pages) std::this_thread::yield();
    // The caller alone looks for the first piece for as long as it takes; the
    // others wait a short time awake (being woken takes about 50 us), then asleep.
    if (caller) {
      (void)wait(0, 0);
      begin();
    }
    for (int i = 0; i < kAwakePolls && !open.load(std::memory_order_acquire); ++i)
      __builtin_ia32_pause();
    if (!open.load(std::memory_order_acquire)) {
      std::unique_lock<std::mutex> g(gate);
      gate_cv.wait(g, [this] { return open.load(std::memory_order_acquire); });
    }
    const size_t per = batch / kPiece;
    for (;;) {
      const size_t i = next.fetch_add(1, std::memory_order_relaxed), b = i / per, k = i % per;
      if (b >= batches() || failed()) return;
      const size_t n = batch_bytes(b), off = k * kPiece;
      if (off >= n) continue;
      if (!wait(b, k)) return;
      memcpy(host + b * batch + off, staging + (b & 1) * half + off,
             n - off < kPiece ? n - off : kPiece);
      if (left[b].fetch_sub(1, std::memory_order_acq_rel) == 1 && b + 2 < batches())
        launch(b + 2);
    }
  }
};

// Runs job.work(whether this is the caller's) on up to `threads` threads, the
// caller's among them.
template <class Job>
static void run_threads(Job& job, int threads) {
  std::vector<std::thread> pool;
  try {
    for (int t = 1; t < threads; ++t)
      pool.emplace_back([&job] {
        if (job.ok(hipSetDevice(job.device))) job.work(false);
      });
  } catch (...) {  // fewer threads than asked for
  }
  job.work(true);
  for (std::thread& t : pool) t.join();
}

static int copy_out(void* host, const void* dev, size_t bytes, void* staging,
                    size_t staging_bytes, uint32_t* flags, uint32_t* count, int threads,
                    hipStream_t st) {
  const std::unique_lock<std::mutex> turn(staging_turn(staging, false), std::try_to_lock);
  if (!turn.owns_lock()) {
    OZK_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st));
    OZK_HIP(hipStreamSynchronize(st));
    return OZK_OK;
  }
  const size_t half = staging_bytes / 2;
  const bool one = bytes <= staging_bytes;
  OutJob job(one ? 1 : (bytes + half - 1) / half);
  job.host = (char*)host;
  job.dev = (const char*)dev;
  job.bytes = bytes;
  job.batch = one ? staging_bytes : half;
  job.half = half;
  job.staging = (char*)staging;
  job.flags = flags;
  job.count = count;
  job.st = st;
  OZK_HIP(hipGetDevice(&job.device));
  for (size_t b = 0; b < job.batches(); ++b) {
    job.seq[b].store(0, std::memory_order_relaxed);
    job.left[b].store((int)((job.batch_bytes(b) + kPiece - 1) / kPiece),
                      std::memory_order_relaxed);
  }
  for (size_t b = 0; b < job.batches() && b < 2; ++b) job.launch(b);
  const size_t pieces = (bytes + kPiece - 1) / kPiece;
  run_threads(job, (size_t)threads < pieces ? threads : (int)pieces);
  if (job.failed()) {
    // nothing of this call may still write the pinned memory
    (void)hipStreamSynchronize(st);
    OZK_HIP((hipError_t)job.err.load());
    set_error("staged copy: the stream is idle and a piece never came");
    return OZK_ERR_HIP;
  }
  g_copied_out.store(st, std::memory_order_relaxed);
  return OZK_OK;
}

// ---------------------------------------------------------------- slots
struct SlotJob {
  bool down;
  char* host;
  char* dev;
  size_t bytes;
  char* staging;
  size_t slot;
  int slots, first;
  void* const* ev;
  hipStream_t st;
  int device;
  std::atomic<size_t> next{0};                // next piece
  std::vector<std::atomic<int>> issued, left;  // per chunk: its copy is queued; pieces to go
  std::atomic<int> err{0};

  explicit SlotJob(size_t n) : issued(n), left(n) {}
  size_t chunks() const { return issued.size(); }
  char* slot_ptr(size_t c) const { return staging + (first + c) % slots * slot; }
  hipEvent_t event(size_t c) const { return (hipEvent_t)ev[(first + c) % slots]; }
  size_t chunk_bytes(size_t c) const {
    return c + 1 < chunks() ? slot : bytes - (chunks() - 1) * slot;
  }
  bool ok(hipError_t e) {
    if (e == hipSuccess) return true;
    int none = 0;
    err.compare_exchange_strong(none, (int)e);
    return false;
  }
  // Queues chunk c's copy, its slot being staged (up) or free (down).
  void issue(size_t c) {
    char *const d = dev + c * slot, *const s = slot_ptr(c);
    if (ok(hipMemcpyAsync(down ? s : d, down ? d : s, chunk_bytes(c),
                          down ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice, st)))
      ok(hipEventRecord(event(c), st));
    issued[c].store(1, std::memory_order_release);
  }
  // Until chunk c's copy is queued; false when something failed.
  bool queued(size_t c) {
    while (!issued[c].load(std::memory_order_acquire)) {
      if (err.load(std::memory_order_relaxed)) return false;
      std::this_thread::yield();
    }
    return !err.load(std::memory_order_relaxed);
  }
  // Pieces in order until none is left or something failed.
  void work(bool) {
    const size_t per = slot / kPiece;
    for (;;) {
      const size_t i = next.fetch_add(1, std::memory_order_relaxed), c = i / per;
      if (c >= chunks() || err.load(std::memory_order_relaxed)) return;
      const size_t off = i % per * kPiece, n = chunk_bytes(c);
      if (off >= n) continue;
      char* const h = host + c * slot + off;
      char* const s = slot_ptr(c) + off;
      const size_t len = n - off < kPiece ? n - off : kPiece;
      if (down) {
        for (size_t b = 0; b < len; b += 4096) ((volatile char*)h)[b] = 0;  // its pages, early
        if (!queued(c) || !ok(hipEventSynchronize(event(c)))) return;
        memcpy(h, s, len);
        if (left[c].fetch_sub(1, std::memory_order_acq_rel) == 1 && c + slots < chunks())
          issue(c + slots);
        continue;
      }
      // the slot's copy before this one has read it: this call's (queued by
      // then), or an earlier call's
      if (c >= (size_t)slots && !queued(c - slots)) return;
      if (!ok(hipEventSynchronize(event(c)))) return;
      memcpy(s, h, len);
      if (left[c].fetch_sub(1, std::memory_order_acq_rel) == 1) issue(c);
    }
  }
};

static int copy_slots(int way, void* dev, void* host, size_t bytes, void* staging,
                      size_t slot_bytes, int slots, int first, void* const* events, int threads,
                      hipStream_t st) {
  if (way != OZK_COPY_UP_NEXT) OZK_HIP(drain(st));
  const std::lock_guard<std::mutex> turn(staging_turn(staging, true));
  SlotJob job((bytes + slot_bytes - 1) / slot_bytes);
  job.down = way == OZK_COPY_DOWN;
  job.host = (char*)host;
  job.dev = (char*)dev;
  job.bytes = bytes;
  job.staging = (char*)staging;
  job.slot = slot_bytes;
  job.slots = slots;
  job.first = first;
  job.ev = events;
  job.st = st;
  OZK_HIP(hipGetDevice(&job.device));
  for (size_t c = 0; c < job.chunks(); ++c) {
    job.issued[c].store(0, std::memory_order_relaxed);
    job.left[c].store((int)((job.chunk_bytes(c) + kPiece - 1) / kPiece),
                      std::memory_order_relaxed);
  }
  for (size_t c = 0; job.down && c < job.chunks() && c < (size_t)slots; ++c) {
    job.ok(hipEventSynchronize(job.event(c)));  // an earlier call's copy
    job.issue(c);
  }
  const size_t pieces = (bytes + kPiece - 1) / kPiece;
  run_threads(job, (size_t)threads < pieces ? threads : (int)pieces);
  if (job.err.load()) {
    // nothing of this call may still use the slots
    (void)hipStreamSynchronize(st);
    OZK_HIP((hipError_t)job.err.load());
  }
  return OZK_OK;
}

// Pinned memory is used again by later calls and a result is waited for, so
// neither copy can be part of a captured graph.
static int refuse_capture(hipStream_t st) {
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  OZK_HIP(hipStreamIsCapturing(st, &cap));
  if (cap == hipStreamCaptureStatusNone) return OZK_OK;
  set_error("a staged copy cannot be captured");
  return OZK_ERR_HIP;
}

}  // namespace ozk

using namespace ozk;

extern "C" {

int ozk_copy_to_host(void* host, const void* dev, size_t bytes, void* staging,
                     size_t staging_bytes, uint32_t* flags, uint32_t* zero_counts, int threads,
                     void* stream) {
  clear_error();
  OZK_CHECK_ARG(threads >= 1 && staging_bytes >= 2 * kPiece && staging_bytes % (2 * kPiece) == 0,
                "staged copy: invalid pinned memory of %zu bytes", staging_bytes);
  if (bytes == 0) return OZK_OK;
  OZK_CHECK_ARG(host && dev && staging && flags && zero_counts, "null pointer");
  const int rc = refuse_capture((hipStream_t)stream);
  if (rc) return rc;
  try {
    return copy_out(host, dev, bytes, staging, staging_bytes, flags, zero_counts, threads,
                    (hipStream_t)stream);
  } catch (const std::exception& e) {
    set_error("staged copy: %s", e.what());
    return OZK_ERR_HIP;
  }
}

int ozk_copy_slots(int way, void* dev, void* host, size_t bytes, void* staging,
                   size_t slot_bytes, int slots, int first, void* const* events, int threads,
                   void* stream) {
  clear_error();
  OZK_CHECK_ARG(way >= OZK_COPY_UP && way <= OZK_COPY_UP_NEXT, "staged copy: way %d", way);
  OZK_CHECK_ARG(slots >= 1 && first >= 0 && threads >= 1 && slot_bytes >= kPiece &&
                    slot_bytes % kPiece == 0,
                "staged copy: invalid ring (%d slots of %zu bytes)", slots, slot_bytes);
  if (bytes == 0) return OZK_OK;
  OZK_CHECK_ARG(host && dev && staging && events, "null pointer");
  const int rc = refuse_capture((hipStream_t)stream);
  if (rc) return rc;
  try {
    return copy_slots(way, dev, host, bytes, staging, slot_bytes, slots, first, events,
                      threads, (hipStream_t)stream);
  } catch (const std::exception& e) {
    set_error("staged copy: %s", e.what());
    return OZK_ERR_HIP;
  }
}

}  // extern "C"
