// Copies of results from HBM to the caller's (pageable) buffers.
//
// hipMemcpyAsync to pageable memory stages through the runtime's own pinned
// buffer, a piece and a wait at a time (16 MB: 0.98 ms).  Here a read is cut
// into pieces that come by DMA (45 GB/s) into a ring of pinned slots, all
// queued at once as far as the ring goes, and go from there to the buffer by
// up to kReaders threads while the next pieces arrive (0.48 ms).  The threads
// matter most where the buffer's pages are new (64 MB of them: 16 ms by one
// thread, 6.4 ms by four).  Whole calls before and after: depths of 64 sources
// on 131 K vertices (8 MB) 760 -> 600 us, three level words of 3.7 M vertices
// (89 MB) 12.4 -> 7.6 ms, 64 searches on Kronecker-22 with one result read
// (32 MB) 17.4 -> 14.6 ms.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

#include "common.h"

namespace dmm {

namespace {

// A piece: an eighth of the read, between these (a DMA takes some 10 us to set
// up: 1.6 MB of a search's results in pieces of 256 KB, 512 KB, 1 MB: 260,
// 224, 209 us for the whole call).  A context holds at most kReadSlots of
// the larger, 16 MB, pinned.
constexpr size_t kPieceLeast = size_t(1) << 20;
constexpr size_t kSmallRead = size_t(512) << 10;  // up to here one wait for all of it
constexpr size_t kPieceMost = size_t(2) << 20;
constexpr size_t kThreadedRead = size_t(2) << 20;       // helpers from here on: starting one costs some 15 us
constexpr int kReaders = 4;

struct Piece {
  char* dst;
  const char* src;
  size_t bytes;
  bool joined;
};

}  // namespace

void read_free(dmm_ctx* ctx) {
  if (ctx->h_ring) (void)hipHostFree(ctx->h_ring);
  ctx->h_ring = nullptr;
  ctx->ring_bytes = 0;
  for (auto& e : ctx->ring_events) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
}

static int read_pieces(dmm_ctx* ctx, const ReadPart* parts, int nparts) {
  size_t total = 0;
  for (int i = 0; i < nparts; i++) total += parts[i].dst ? parts[i].bytes : 0;
  if (total == 0) {
    DMM_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    return DMM_OK;
  }
  const size_t slot =
      std::min(kPieceMost, std::max(kPieceLeast, (total / kReadSlots + (size_t(1) << 16) - 1) >> 16 << 16));
  std::vector<Piece> pieces;
  for (int i = 0; i < nparts; i++) {
    if (!parts[i].dst) continue;
    char* d = static_cast<char*>(parts[i].dst);
    const char* s = static_cast<const char*>(parts[i].src);
    const bool joined = parts[i].joined && i > 0 && parts[i - 1].dst;
    for (size_t o = 0; o < parts[i].bytes; o += slot)
      pieces.push_back({d + o, s + o, std::min(slot, parts[i].bytes - o), joined && o == 0});
  }
  const int n = static_cast<int>(pieces.size());
  // Slot s holds the pieces s, s + slots, ...  The ring grows to what a read
  // can use of it.
  const int slots = std::min(n, kReadSlots);
  if (ctx->ring_bytes < slots * slot) {
    DMM_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    read_free(ctx);
    if (hipHostMalloc(reinterpret_cast<void**>(&ctx->h_ring), slots * slot, hipHostMallocDefault) != hipSuccess) {
      ctx->h_ring = nullptr;
      (void)hipGetLastError();
    } else {
      ctx->ring_bytes = slots * slot;
    }
  }
  for (auto& e : ctx->ring_events)
    if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
      e = nullptr;
      (void)hipGetLastError();
    }
  bool direct = !ctx->h_ring;
  for (auto& e : ctx->ring_events) direct = direct || !e;
  if (direct) {  // no pinned memory to be had: the runtime's own path
    for (int i = 0; i < nparts; i++)
      if (parts[i].dst && parts[i].bytes)
        DMM_HIP_CHECK(ctx, hipMemcpyAsync(parts[i].dst, parts[i].src, parts[i].bytes, hipMemcpyDeviceToHost, ctx->stream));
    DMM_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    return DMM_OK;
  }
  if (total <= kSmallRead) {
    // Joined parts come in one piece.  (That two parts' addresses follow one
    // another does not say so: a copy must not span allocations.)
    size_t at = 0;
    for (int i = 0; i < n;) {
      size_t run = pieces[i].bytes;
      int j = i + 1;
      for (; j < n && pieces[j].joined; j++) run += pieces[j].bytes;
      DMM_HIP_CHECK(ctx, hipMemcpyAsync(ctx->h_ring + at, pieces[i].src, run, hipMemcpyDeviceToHost, ctx->stream));
      at += run;
      i = j;
    }
    DMM_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    at = 0;
    for (const Piece& p : pieces) {
      std::memcpy(p.dst, ctx->h_ring + at, p.bytes);
      at += p.bytes;
    }
    return DMM_OK;
  }
  std::vector<std::atomic<int>> queued(n);  // 1: its DMA and event are on the stream, 2: they could not be
  for (auto& q : queued) q.store(0, std::memory_order_relaxed);
  std::atomic<int> next{0}, error{0};
  auto queue = [&](int i) {
    char* at = ctx->h_ring + (i % slots) * slot;
    hipError_t e = hipMemcpyAsync(at, pieces[i].src, pieces[i].bytes, hipMemcpyDeviceToHost, ctx->stream);
    if (e == hipSuccess) e = hipEventRecord(ctx->ring_events[i % slots], ctx->stream);
    if (e != hipSuccess) error.store(static_cast<int>(e));
    queued[i].store(e == hipSuccess ? 1 : 2, std::memory_order_release);
  };
  // Every piece is taken once; a slot's next piece is queued by the thread
  // that emptied it, so every wait here is for a piece some thread is past.
  auto work = [&] {
    (void)hipSetDevice(ctx->device);
    for (;;) {
      const int i = next.fetch_add(1);
      if (i >= n) return;
      int q;
      while ((q = queued[i].load(std::memory_order_acquire)) == 0) std::this_thread::yield();
      if (q == 1) {
        const hipError_t e = hipEventSynchronize(ctx->ring_events[i % slots]);
        if (e == hipSuccess)
          std::memcpy(pieces[i].dst, ctx->h_ring + (i % slots) * slot, pieces[i].bytes);
        else
          error.store(static_cast<int>(e));
      }
      if (i + slots < n) queue(i + slots);
    }
  };
  for (int i = 0; i < slots; i++) queue(i);
  std::thread helpers[kReaders - 1];
  if (total >= kThreadedRead) {
    for (int k = 0; k < kReaders - 1; k++) {
      try {
        helpers[k] = std::thread(work);
      } catch (const std::system_error&) {
        break;  // the caller reads alone
      }
    }
  }
  work();
  for (auto& t : helpers)
    if (t.joinable()) t.join();
  if (error.load()) {
    (void)hipStreamSynchronize(ctx->stream);
    return set_err(ctx, DMM_ERR_HIP, "reading results failed: %s", hipGetErrorString(static_cast<hipError_t>(error.load())));
  }
  return DMM_OK;
}

int read_out(dmm_ctx* ctx, const ReadPart* parts, int nparts) {
  try {
    return read_pieces(ctx, parts, nparts);
  } catch (const std::bad_alloc&) {  // before anything is queued
    return set_err(ctx, DMM_ERR_NOMEM, "host allocation for a read failed");
  }
}

}  // namespace dmm
