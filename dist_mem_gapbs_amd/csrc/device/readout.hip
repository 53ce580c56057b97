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
constexpr size_t kThreadedRead = size_t(2) << 20;  // helpers from here on: starting one costs some 15 us; also on new pages
// A ring that is too small for a read: pieces of a quarter of it, for this many
// reads.  After them it grows, beside the levels where there are some.  A whole
// batch of 64 sources, the first through the search's ring, the second, the one
// that enlarges it, later ones: 20 K vertices (1.3 MB) 389, 251, 489, 188 us; 131
// K (8.4 MB) 952, 621, 1512, 450; enlarged by the upload 419, 254, 197 and 1405,
// 506, 450, and the uploads 0.4 and 0.3 ms longer.
constexpr int kShortSlots = 4;
constexpr int kShortReads = 2;
static_assert(kShortSlots <= kReadSlots, "flags");
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
  if (ctx->h_ring_old) (void)hipHostFree(ctx->h_ring_old);
  ctx->h_ring = ctx->h_ring_old = nullptr;
  ctx->ring_bytes = 0;
}

// A ring of `bytes` of slots in place of a smaller one, which stays in use if
// there is no pinned memory to be had, and is freed with the next one replaced
// otherwise (65 us, which is not for this read).
static void ring_alloc(dmm_ctx* ctx, size_t bytes) {
  char* ring = nullptr;
  if (hipHostMalloc(reinterpret_cast<void**>(&ring), kFlagBytes + bytes, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    return;
  }
  std::memset(ring, 0, kFlagBytes);
  if (ctx->h_ring_old) (void)hipHostFree(ctx->h_ring_old);
  ctx->h_ring_old = ctx->h_ring;
  ctx->h_ring = ring;
  ctx->ring_bytes = bytes;
  ctx->ring_touched = 0;
  ctx->short_reads = 0;
  ctx->read_seq = 0;
}

// The slots of a read: an eighth of it each, between the least and the most.
static size_t slot_bytes(size_t total) {
  return std::min(kPieceMost, std::max(kPieceLeast, (total / kReadSlots + (size_t(1) << 16) - 1) >> 16 << 16));
}

static size_t total_bytes(const ReadPart* parts, int nparts) {
  size_t total = 0;
  for (int i = 0; i < nparts; i++) total += parts[i].dst ? parts[i].bytes : 0;
  return total;
}

// The ring that a read can use.
static size_t ring_of(const ReadPart* parts, int nparts) {
  const size_t slot = slot_bytes(total_bytes(parts, nparts));
  size_t slots = 0;
  for (int i = 0; i < nparts; i++) slots += parts[i].dst ? (parts[i].bytes + slot - 1) / slot : 0;
  return std::min<size_t>(slots, kReadSlots) * slot;
}

ReadWarm::ReadWarm(dmm_ctx* ctx, int64_t rows) {
  // A parent and a depth; an FP64 rank needs no more.
  const size_t bytes = sizeof(int32_t) * static_cast<size_t>(rows);
  const ReadPart search[] = {{ctx, nullptr, bytes}, {ctx, nullptr, bytes}};
  start(ctx, ring_of(search, 2));
}

ReadWarm::ReadWarm(dmm_ctx* ctx, const ReadPart* parts, int nparts) {
  if (ctx->short_reads >= kShortReads) start(ctx, ring_of(parts, nparts));
}

void ReadWarm::start(dmm_ctx* ctx, size_t want) {
  if (ctx->ring_bytes >= want) return;
  // Without a thread the read allocates.
  (void)start_thread(&thread, [this, ctx, want] {
    (void)hipSetDevice(ctx->device);
    ring_alloc(ctx, want);
    if (ctx->ring_bytes < want) return;
    size_t i = 0;
    for (; i < want && !done.load(std::memory_order_relaxed); i += 4096)
      reinterpret_cast<volatile char*>(ctx->h_ring)[kFlagBytes + i] = 0;
    ctx->ring_touched = i;
  });
}

ReadWarm::~ReadWarm() {
  done.store(true, std::memory_order_relaxed);
  if (thread.joinable()) thread.join();
}

static int read_pieces(dmm_ctx* ctx, const ReadPart* parts, int nparts) {
  const size_t total = total_bytes(parts, nparts);
  if (total == 0) {
    DMM_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    return DMM_OK;
  }
  std::vector<Piece> pieces;
  auto cut = [&](size_t slot) {
    pieces.clear();
    for (int i = 0; i < nparts; i++) {
      if (!parts[i].dst) continue;
      char* d = static_cast<char*>(parts[i].dst);
      const char* s = static_cast<const char*>(parts[i].src);
      for (size_t o = 0; o < parts[i].bytes; o += slot)
        pieces.push_back({d + o, s + o, std::min(slot, parts[i].bytes - o)});
    }
    return static_cast<int>(pieces.size());
  };
  // Slot s holds the pieces s, s + slots, ...  The ring grows to what a read
  // can use of it, but not for the first few that it is too small for, nor for
  // one that smaller pieces get through it at once.
  size_t slot = slot_bytes(total);
  int n = cut(slot);
  int slots = std::min(n, kReadSlots);
  if (ctx->ring_bytes < slots * slot) {
    const size_t whole = slots * slot;
    const auto quarters = [&] {
      slot = ctx->ring_bytes / kShortSlots / 4096 * 4096;
      n = cut(slot);
      slots = std::min(n, kShortSlots);
    };
    if (ctx->ring_bytes > 0) quarters();
    if (ctx->ring_bytes == 0 || (n > slots && ++ctx->short_reads > kShortReads)) {
      DMM_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
      ring_alloc(ctx, whole);
      if (ctx->ring_bytes >= whole) {
        slot = slot_bytes(total);
        n = cut(slot);
        slots = std::min(n, kReadSlots);
      }
    }
  }
  if (ctx->ring_bytes == 0) {  // no pinned memory to be had: the runtime's own path
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
  const bool each = total > kSmallRead || n > slots;
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
  const size_t used = slots * slot;
  if (total >= kThreadedRead || (each && used > ctx->ring_touched)) {
    for (int k = 0; k < kReaders - 1; k++)
      if (!start_thread(&helpers[k], work)) break;  // those that there are read alone
  }
  work();
  for (auto& t : helpers)
    if (t.joinable()) t.join();
  ctx->ring_touched = std::max(ctx->ring_touched, used);
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
