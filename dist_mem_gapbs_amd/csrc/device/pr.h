// Launchers of the pull PageRank kernels (pr.hip).
#ifndef DMM_DEVICE_PR_H_
#define DMM_DEVICE_PR_H_

#include <memory>
#include <string>
#include <utility>
#include <vector>

#include "common.h"

namespace dmm {

// Work items of the compensated / FP64 modes: a heavy row (slot < 0) or one
// segment of a split row (its partial goes to partial[slot]).
struct PrItem {
  int32_t v;
  int32_t slot;
  int64_t b, e;
};
// A split row: its segments' partials are partial[first .. first + count).
struct PrSuper {
  int32_t v;
  int32_t first;
  int32_t count;
  int32_t pad;
};
constexpr int64_t kPrSplit = 2048;    // rows with more in-edges are split
constexpr int64_t kPrSegment = 2048;  // edges per segment

// Serial mode: work items (dealt to workgroups at upload).  A bundle of 16
// rows of 1023 edges is the longest item of a small graph when rows go to
// wavefronts from 1024 on: a whole Kronecker-14 rank takes 305 us with 512
// and 372 us with 1024 (Kronecker-21 2.42 and 2.35 ms; 256: no change).  A
// wavefront gathers some 0.1 G/s beside others, so the longest rows need a
// workgroup: Kronecker-21 2.42 ms from 32768 (or 16384) on, 2.72 from 131072.
constexpr int64_t kSerialWaveRow = 512;     // rows from here on: a wavefront each
constexpr int64_t kSerialBlockRow = 32768;  // rows from here on: a workgroup each
// ... in a small graph: halved down to this while the CUs would have less than
// such a row each (200 K vertices, 20 iterations: 816 us; 936 from 32768 on;
// least 1024 or 4096: no change).
constexpr int64_t kSerialBlockLeast = 2048;
constexpr int kHeavyBundle = 16;            // shorter heavy rows: this many per wavefront
constexpr int kLightBundle = 64;            // rows below the heavy threshold
enum : int32_t {
  kSerialBlock = 0,  // row `first`, by the workgroup
  kSerialWave = 1,   // row `first`, by a wavefront
  kSerialHeavy = 2,  // heavy-list entries [first, first + kHeavyBundle)
  kSerialLight = 3,  // the light ones of rows [first, first + kLightBundle)
};
struct SerialItem {
  int32_t first;
  int32_t kind;
};
void serial_plan(int64_t rows, int64_t light_begin, int64_t zero_begin, const int64_t* off,
                 const std::vector<int32_t>& heavy, const std::vector<int32_t>& by_class, int blocks,
                 std::vector<SerialItem>* items, std::vector<int32_t>* start);

// Window-tiled compensated PageRank (degree-ordered whole graphs).
// Sources are cut into windows of `pr_window` vertices (a tuning value:
// 16384 or 32768 contributions, 64 or 128 KB of LDS).  Every in-edge sits
// in a 64-lane chunk of its source's window, kLaneEdges edges per lane, and
// is summed from an LDS copy of that window; each piece (a row's edges
// inside one chunk) leaves one partial, its FP64 sum rounded to FP32, and
// the row kernel merges a row's partials in window order.
constexpr int kLaneEdges = 16;
constexpr int kChunkEdges = 64 * kLaneEdges;
constexpr int kChunkPieces = 512;   // pieces one chunk may hold
// Row blocks: consecutive rows holding at most kBlockRuns runs; rows with
// kSoloRuns runs or kSoloEdges in-edges or more are blocks of their own.
// A block's partials (its runs plus chunk cuts) must number at most
// kRowSlots: the row kernel gathers them into LDS.
constexpr int kRowSlots = 8192;
constexpr int kRowThreads = 512;    // threads of the row kernel
constexpr int kRowGroupsPerCU = 4;  // row kernel workgroups resident per CU
constexpr int kBlockRuns = 6144;
constexpr int kSoloRuns = 256;
constexpr int64_t kSoloEdges = 4096;

// The tile layout as built on the host.  Partials are numbered window-major
// in chunk order (chunk c writes [cbase[c], cbase[c + 1])); a row block's
// partials in one window are contiguous there (a segment), and its region
// is the concatenation of its segments in window order.
struct TileHost {
  std::vector<int32_t> cwin;     // window of each chunk
  std::vector<int64_t> wstart;   // first chunk of each window (+ end)
  std::vector<int32_t> cbase;    // first partial of each chunk (+ end)
  std::vector<uint32_t> meta;    // per lane: end mask (bit j: slot j ends a piece) | filled slots << 16
  std::vector<uint16_t> src;     // kChunkEdges per chunk
  std::vector<int32_t> brow;     // row blocks: first row (+ end)
  std::vector<int64_t> bseg;     // row blocks: first segment (+ end)
  std::vector<int32_t> bsize;    // row blocks: partials (the region's size)
  std::vector<int32_t> seg_start;  // segments: first partial
  std::vector<int32_t> seg_off;    //           offset in the block's region
  std::vector<int32_t> istart;   // rows [0, zb]: first list entry (rows of one-row blocks have none)
  std::vector<uint16_t> idx;     // per row, window order: partial offsets in its block's region
  int64_t n_pieces = 0, slots_filled = 0, window = 0;
  int32_t n_windows = 0;
};

// Builds the tile layout of an in-CSR (n rows, sources in [0, n_gather),
// rows at and above zb without in-edges); sorts nbr row by row in place.
int build_tiles_host(int64_t n, int64_t zb, int64_t n_gather, const int64_t* off, int32_t* nbr, int64_t window,
                     TileHost* out, std::string* err);

// Builds the tiled structures from the device CSR (host work, once per
// upload, at the first compensated call).  Returns DMM_OK or an error.
int pr_tiles_build(dmm_ctx* ctx);

// Compensated PageRank of a PE block (rows in the caller's order, sources
// anywhere in the whole graph): propagation layout.  Pass 1 copies one
// window of kBWin contributions into LDS at a time and writes each in-edge's
// contribution to the edge's place in the bucket-major array; pass 2 sums
// each bucket's rows exactly, as 128-bit fixed-point integers.  Two bucket
// shapes:
//   fine    a bucket's contributions fit LDS: pass 2 sorts them there by row
//           (static places) and sums each row's run in registers
//   coarse  a bucket's row accumulators fit LDS: pass 2 adds every
//           contribution with LDS atomics, at about 350 G/s, and a block that
//           does not fill the CUs with buckets of 2^19 edges waits for the
//           largest.  For blocks with more fine buckets than a window's segment
//           table holds (from some 125 M in-edges or 16 M rows on), and where
//           the fine buckets' shorter segments cost more (fine_is_faster).
//           Kronecker-23, block 3 of 8, pass 1 + pass 2: coarse 52 + 281 us,
//           fine 61 + 75 us.
constexpr int kBWin = 32768;             // sources per window (128 KB of LDS)
struct BlockShape {
  int64_t rows;   // rows per bucket
  int64_t edges;  // in-edges per bucket, and per unit of a one-row bucket
  bool fine;
};
constexpr int kBRows = 8192;             // coarse: the accumulators fill 128 KB of LDS
constexpr int64_t kBEdges = 1 << 19;
constexpr int kFineRows = 2048;
constexpr int kFineEdges = 16384;        // with the row sums 72 KB of LDS: two workgroups per CU
constexpr int kFineLeast = 1024;         // ... of a small block, so that its buckets reach more CUs
constexpr int kFineLong = 256;           // rows from here on are summed by the workgroup,
constexpr int kFineMid = 8;              // from here on by eight lanes, shorter ones by a thread
constexpr BlockShape kCoarse = {kBRows, kBEdges, false};
constexpr BlockShape kFine = {kFineRows, kFineEdges, true};
constexpr int kBSegMax = 8000;           // buckets a window's segment table may hold (beside the window in LDS)
constexpr int kBPer = 8;                 // edges per thread in pass 1 (window starts padded to it)
struct BlockUnit {  // pass 2 work: bucket rows [row0, row0 + nrows), edges [e0, e1)
  int32_t row0;
  int32_t nrows;
  int32_t slot;  // >= 0: a part of a one-row bucket, its sum goes to partial slot `slot`
  int32_t nlong; // fine: rows of kFineLong in-edges and more (the first in its part of `rows`)
  int32_t nmid;  // ... of kFineMid and more
  int32_t pad;
  int64_t e0, e1;
};
struct BlockGroup {   // 64 consecutive edges of a window
  uint64_t starts;    // bit k: edge k + 1 of the group begins a segment
  int32_t first;      // the segment, in the window, of the group's edge 0
  int32_t pad;
};
struct FineRow {  // row `row` of a fine bucket: places [start, start + len)
  uint16_t row, start, len, pad;
};
struct BlockSplit {  // a one-row bucket in parts: partial slots [first, first + count)
  int32_t row;
  int32_t first;
  int32_t count;
  int32_t pad;
};
// An array whose elements hold nothing until they are written.
template <typename T>
class RawArray {
 public:
  RawArray() = default;
  explicit RawArray(int64_t n) : p_(new T[static_cast<size_t>(n)]), n_(static_cast<size_t>(n)) {}
  T& operator[](int64_t i) { return p_[i]; }
  const T& operator[](int64_t i) const { return p_[i]; }
  T* data() { return p_.get(); }
  const T* data() const { return p_.get(); }
  size_t size() const { return n_; }
  void swap(RawArray& o) {
    p_.swap(o.p_);
    std::swap(n_, o.n_);
  }

 private:
  std::unique_ptr<T[]> p_;
  size_t n_ = 0;
};
struct BlockHost {
  RawArray<uint16_t> src;          // window-major source offsets (window starts padded to kBPer)
  std::vector<int64_t> wstart;     // window starts (+ end)
  std::vector<int32_t> wlen;       // window edge counts
  std::vector<int64_t> wseg;       // first segment of each window (+ end)
  RawArray<int32_t> seg_e;         // segment start inside its window
  RawArray<int32_t> seg_d;         // segment destination minus seg_e
  std::vector<int64_t> wgroup;     // first group of 64 edges of each window (+ end)
  RawArray<BlockGroup> groups;     // per group: where segments start in it
  RawArray<uint16_t> brow_off;     // bucket-major; coarse: row offset inside the bucket, fine: place, rows by length
  RawArray<FineRow> rows;          // fine: per bucket (from its first row on), longest class first
  std::vector<BlockUnit> units;
  std::vector<BlockSplit> splits;
  int32_t n_slots = 0, n_windows = 0;
  int64_t n_buckets = 0;
};
// Builds the propagation layout of an in-CSR of n rows with sources in
// [0, n_gather) with buckets of the given shape.  Returns DMM_OK or an error
// code (message in *err; DMM_ERR_CAPACITY also for too many buckets).
int build_blocks_host(int64_t n, int64_t n_gather, const int64_t* off, const int32_t* nbr, const BlockShape& shape,
                      BlockHost* out, std::string* err);
// Builds it from the device CSR (host work, once per upload, at the first
// compensated block iteration).
int pr_blocks_build(dmm_ctx* ctx);

int pr_light_blocks(dmm_ctx* ctx);
int pr_serial_blocks(dmm_ctx* ctx);  // workgroups of a serial-mode iteration
int pr_super_blocks(dmm_ctx* ctx);
int pr_fused_blocks(dmm_ctx* ctx);  // persistent KAHAN / FP64 kernel
int pr_row_blocks(dmm_ctx* ctx);    // row kernel of the tiled compensated mode
int pr_bsum_blocks(dmm_ctx* ctx);   // PE-block compensated mode: bucket sums
int pr_bsplit_blocks(dmm_ctx* ctx); //   and the rows summed in parts
// Size of the PrParams block (bytes) the ctx must hold at d_prparams.
constexpr size_t kPrParamsBytes = 64;

int pr_run(dmm_ctx* ctx, int32_t max_iters, double epsilon, int32_t mode, dmm_pr_stats* stats);
int pr_block_iteration(dmm_ctx* ctx, const float* gcontrib_host, float* scores_inout, int32_t mode,
                       double* err, double* ms);
// The context's device address of this GPU's scratch array (once per
// device), kept in ctx->scratch.
int scratch_init(dmm_ctx* ctx);
// pr_block_iteration on device buffers with every temporary in the scratch
// array: no device allocation.
int pr_block_iteration_noalloc(dmm_ctx* ctx, const float* d_gcontrib, float* d_scores, float* d_contrib_out,
                               int32_t mode, double* d_err);

}  // namespace dmm

#endif  // DMM_DEVICE_PR_H_
