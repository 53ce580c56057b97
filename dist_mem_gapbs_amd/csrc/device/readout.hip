// Copies of results from HBM to the caller's (pageable) buffers.
//
// hipMemcpyAsync to pageable memory stages through the runtime's own pinned
// buffer, a piece and a wait at a time (16 MB: 0.98 ms).  Here a read is cut
// into pieces that a kernel stores into a ring of pinned slots, as far as the
// ring goes in one launch; up to kReaders threads carry them to the buffer
// while the next pieces arrive.  The threads matter most where the buffer's
// pages are new (64 MB of them: 16 ms by one thread, 6.4 ms by four).
#include <algorithm>
#include <atomic>
#include <cstring>
#include <new>
#include <thread>
#include <vector>

#include "../host/threads.h"
#include "common.h"

namespace dmm {

namespace {

// A piece: an eighth of the read, between these.  A context holds at most
// kReadSlots of the larger, 16 MB, pinned.
constexpr size_t kPieceLeast = size_t(256) << 10;
constexpr size_t kPieceMost = size_t(2) << 20;
constexpr size_t kSmallRead = size_t(512) << 10;    // up to here one wait for all of it
constexpr size_t kThreadedRead = size_t(2) << 20;  // helpers from here on: starting one costs some 15 us
constexpr int kReaders = 4;
constexpr int64_t kGroupLeast = int64_t(16) << 10;  // of a small read, by each workgroup
constexpr int kThreads = 256;
constexpr int kUnroll = 4;
constexpr size_t kFlagBytes = 4096;  // the slots behind them start on a page
static_assert(sizeof(uint32_t) * kReadSlots * kReadGroups <= kFlagBytes, "flags of every workgroup and slot");

struct Piece {
  char* dst;
  const char* src;
  size_t bytes;
};

struct ReadList {
  const char* src[kReadSlots];
  uint32_t bytes[kReadSlots];
};

// n pieces into the slots from `slot` on, one after the other, each by all
// workgroups.  Bound by the link (PCIe, 56 GB/s).  A workgroup whose part of a
// piece has been stored says so in its own pinned flag, so a piece needs
// neither an event nor a copy command of its own: with those, every 2 MB
// (37 us) were followed by 10 us in which nothing moved.  each: every piece
// has its flags, else the last, for all.  Copy commands, then this: depths of
// 64 sources on 131 K vertices (8 MB) 541 -> 448 us a call, path counts of
// 480 K vertices (9.6 MB) 553 -> 467, a search's 32 MB 902 -> 780 (the read);
// up to 512 KB the same.  16, 32, 64, 128 workgroups: 453, 448, 461, 490 us.
__global__ __launch_bounds__(kThreads) void k_read(ReadList l, int n, char* slot, size_t slot_bytes, uint32_t* flags,
                                                   uint32_t seq, bool each) {
  const uint32_t t = blockIdx.x * kThreads + threadIdx.x;
  const uint32_t step = gridDim.x * kThreads;
  for (int p = 0; p < n; p++, slot += slot_bytes, flags += kReadGroups) {
    const char* __restrict__ src = l.src[p];
    const uint32_t words = l.bytes[p] / 16;
    uint4* out = reinterpret_cast<uint4*>(slot);
    for (uint32_t i = t; i < words; i += kUnroll * step) {
      uint4 v[kUnroll];
#pragma unroll
      for (int j = 0; j < kUnroll; j++)  // a part may start at any byte
        __builtin_memcpy(&v[j], src + size_t(min(i + j * step, words - 1)) * 16, 16);
#pragma unroll
      for (int j = 0; j < kUnroll; j++)
        if (i + j * step < words) out[i + j * step] = v[j];
    }
    const uint32_t tail = words * 16 + t;
    if (tail < l.bytes[p]) slot[tail] = src[tail];
    if (!each && p + 1 < n) continue;
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0)
      __hip_atomic_store(&flags[blockIdx.x], seq + p, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

}  // namespace

void read_free(dmm_ctx* ctx) {
  if (ctx->h_ring) (void)hipHostFree(ctx->h_ring);
  ctx->h_ring = nullptr;
  ctx->ring_bytes = 0;
}

// A ring of `bytes` of slots (none if there is no pinned memory to be had).
static void ring_alloc(dmm_ctx* ctx, size_t bytes) {
  read_free(ctx);
  if (hipHostMalloc(reinterpret_cast<void**>(&ctx->h_ring), kFlagBytes + bytes, hipHostMallocDefault) != hipSuccess) {
    ctx->h_ring = nullptr;
    (void)hipGetLastError();
    return;
  }
  ctx->ring_bytes = bytes;
  std::memset(ctx->h_ring, 0, kFlagBytes);
  ctx->read_seq = 0;
}

ReadWarm::ReadWarm(dmm_ctx* ctx, int64_t rows) {
  const size_t search = 8 * static_cast<size_t>(rows);  // a parent and a depth, or an FP64 rank
  // A larger ring is an allocation of its own in the driver, which holds up
  // the upload's: no more than a search needs where that is a small read (a
  // batch then enlarges it), else what a batch can use of it.
  const size_t want = search <= kSmallRead
                          ? 2 * kPieceLeast
                          : std::min(kReadSlots * kPieceMost, 8 * search + kReadSlots * (size_t(1) << 16));
  if (ctx->ring_bytes >= want) return;
  const size_t touch = std::min(want, std::max(2 * kThreadedRead, 2 * search));
  // Without a thread the first read allocates.
  (void)start_thread(&thread, [this, ctx, want, touch] {
    (void)hipSetDevice(ctx->device);
    ring_alloc(ctx, want);
    if (!ctx->h_ring) return;
    for (size_t i = 0; i < touch && !done.load(std::memory_order_relaxed); i += 4096)
      reinterpret_cast<volatile char*>(ctx->h_ring)[kFlagBytes + i] = 0;
  });
}

ReadWarm::~ReadWarm() {
  done.store(true, std::memory_order_relaxed);
  if (thread.joinable()) thread.join();
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
    for (size_t o = 0; o < parts[i].bytes; o += slot) pieces.push_back({d + o, s + o, std::min(slot, parts[i].bytes - o)});
  }
  const int n = static_cast<int>(pieces.size());
  // Slot s holds the pieces s, s + slots, ...  The ring grows to what a read
  // can use of it.
  const int slots = std::min(n, kReadSlots);
  if (ctx->ring_bytes < slots * slot) {
    DMM_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    ring_alloc(ctx, slots * slot);
  }
  if (!ctx->h_ring) {  // no pinned memory to be had: the runtime's own path
    for (int i = 0; i < nparts; i++)
      if (parts[i].dst && parts[i].bytes)
        DMM_HIP_CHECK(ctx, hipMemcpyAsync(parts[i].dst, parts[i].src, parts[i].bytes, hipMemcpyDeviceToHost, ctx->stream));
    DMM_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    return DMM_OK;
  }
  uint32_t* const flags = reinterpret_cast<uint32_t*>(ctx->h_ring);
  char* const ring = ctx->h_ring + kFlagBytes;
  // Piece i is there once its slot's flags hold seq + i; no other piece of
  // the slot before or after it has that number.
  if (ctx->read_seq > UINT32_MAX - static_cast<uint32_t>(n) - 1) {
    DMM_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    std::memset(flags, 0, kFlagBytes);
    ctx->read_seq = 0;
  }
  const bool each = total > kSmallRead;
  const int groups = each ? kReadGroups : static_cast<int>(std::min<size_t>(kReadGroups, ceil_div(total, kGroupLeast)));
  const uint32_t seq = ctx->read_seq + 1;
  ctx->read_seq += static_cast<uint32_t>(n);
  std::vector<std::atomic<int>> queued(n);  // 1: its copy is on the stream, 2: it could not be
  for (auto& q : queued) q.store(0, std::memory_order_relaxed);
  std::atomic<int> next{0}, error{0};
  auto queue = [&](int i, int count) {
    ReadList l{};
    for (int k = 0; k < count; k++) {
      l.src[k] = pieces[i + k].src;
      l.bytes[k] = static_cast<uint32_t>(pieces[i + k].bytes);
    }
    const int s = i % slots;
    hipLaunchKernelGGL(k_read, dim3(groups), dim3(kThreads), 0, ctx->stream, l, count, ring + s * slot, slot,
                       flags + s * kReadGroups, seq + static_cast<uint32_t>(i), each);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) error.store(static_cast<int>(e));
    for (int k = 0; k < count; k++) queued[i + k].store(e == hipSuccess ? 1 : 2, std::memory_order_release);
  };
  auto stored = [&](int i) {
    const uint32_t* f = flags + (i % slots) * kReadGroups;
    for (int g = 0; g < groups; g++)
      if (__atomic_load_n(&f[g], __ATOMIC_ACQUIRE) != seq + static_cast<uint32_t>(i)) return false;
    return true;
  };
  // A stream that has ended, well or not, without the flags set ends the wait.
  auto wait = [&](int i) -> hipError_t {
    for (int spins = 1;; spins++) {
      if (stored(i)) return hipSuccess;
      if (spins % 65536 == 0) {
        const hipError_t e = hipStreamQuery(ctx->stream);
        if (e == hipErrorNotReady) {
          (void)hipGetLastError();
          std::this_thread::yield();
        } else if (!stored(i)) {
          return e == hipSuccess ? hipErrorUnknown : e;
        }
      }
    }
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
        const hipError_t e = wait(each ? i : n - 1);
        if (e == hipSuccess)
          std::memcpy(pieces[i].dst, ring + (i % slots) * slot, pieces[i].bytes);
        else
          error.store(static_cast<int>(e));
      }
      if (i + slots < n) queue(i + slots, 1);
    }
  };
  queue(0, slots);
  std::thread helpers[kReaders - 1];
  if (total >= kThreadedRead) {
    for (int k = 0; k < kReaders - 1; k++)
      if (!start_thread(&helpers[k], work)) break;  // those that there are read alone
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
