// Host-side construction of the propagation layout of a PE block's
// compensated PageRank iteration (the block's rows in the caller's order,
// sources anywhere in [0, n_gather)).
//
// Sources are cut into windows of kBWin vertices (one window of
// contributions fills a workgroup's LDS); rows into buckets of at most
// shape.rows consecutive rows and shape.edges in-edges (a row with more
// in-edges is a bucket of its own, summed in units of at most that many).
// Edge (u -> r) belongs to segment (window u / kBWin, bucket of r).
//
//   window-major array (pass 1 reads it): per window its edges' 16-bit
//     source offsets, segment by segment in bucket order, the window's
//     start padded to a multiple of kBPer edges;
//   bucket-major array (pass 1 writes it, pass 2 reads it): per bucket its
//     edges' contributions, segment by segment in window order, and beside
//     it (static) each edge's row offset inside its bucket (coarse) or its
//     place among the bucket's edges, rows by length (fine).
// The i-th edge of a segment sits at the i-th place of the segment in both
// arrays.  Per window, the segment table gives each non-empty segment's
// destination in the bucket-major array (stored as destination - start, so an
// edge's destination is that plus its index in the window), and per group of
// 64 edges of the window a mask says where segments start, so that a lane
// counts its segment instead of searching for it.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../host/parallel.h"
#include "pr.h"

namespace dmm {

namespace {

// Buckets of the shape: their first rows (+ end).
std::vector<int32_t> cut_buckets(int64_t n, const int64_t* off, const BlockShape& shape) {
  std::vector<int32_t> brow{0};
  int64_t rows = 0, edges = 0;
  for (int64_t r = 0; r < n; r++) {
    const int64_t d = off[r + 1] - off[r];
    if (rows > 0 && (rows == shape.rows || edges + d > shape.edges)) {
      brow.push_back(static_cast<int32_t>(r));
      rows = edges = 0;
    }
    rows++;
    edges += d;
  }
  if (n > 0) brow.push_back(static_cast<int32_t>(n));
  return brow;
}

}  // namespace

// Host time counts: a block's first iteration waits for this.  With many
// windows the (window, bucket) tables are the larger part, so a bucket's entries
// lie together, every pass over them is shared out, and nothing is filled
// before it is written (33 M edges from 2^27 sources, fine: 297 ms for the first
// iteration with window-major tables, serial passes and zeroed vectors).
int build_blocks_host(int64_t n, int64_t n_gather, const int64_t* off, const int32_t* nbr, const BlockShape& shape,
                      BlockHost* out, std::string* err) {
  const int nt = resolve_threads(0);
  const int64_t m = off[n];
  if (m >= (int64_t(1) << 31) || n_gather >= (int64_t(1) << 31)) {
    *err = "PE block too large for the propagation layout";
    return DMM_ERR_CAPACITY;
  }
  const int32_t nwin = static_cast<int32_t>(std::max<int64_t>(1, (n_gather + kBWin - 1) / kBWin));
  // 1. Buckets.
  const std::vector<int32_t> brow = cut_buckets(n, off, shape);
  const int64_t nb = static_cast<int64_t>(brow.size()) - 1;
  if (nb > kBSegMax) {
    *err = "PE block has more row buckets than a window's segment table holds";
    return DMM_ERR_CAPACITY;
  }
  // 2. Bucket-major: a segment's start inside its bucket, boff[b * pitch + w]
  // (+ end).
  const int64_t pitch = int64_t(nwin) + 1;
  RawArray<uint32_t> boff(nb * pitch);
  auto window = [](int32_t u) { return static_cast<uint32_t>(u) / kBWin; };
  parallel_dynamic(nb, nt, 4, [&](int64_t b) {
    uint32_t* o = &boff[b * pitch];
    std::fill(o, o + pitch, 0u);
    for (int64_t e = off[brow[b]]; e < off[brow[b + 1]]; e++) o[window(nbr[e]) + 1]++;
    for (int32_t w = 0; w < nwin; w++) o[w + 1] += o[w];
  });
  std::vector<int64_t> bstart(nb + 1, 0);
  for (int64_t b = 0; b < nb; b++) bstart[b + 1] = off[brow[b + 1]];
  // 3. Window-major: its start inside its window, wrel[b * nwin + w]; a cache
  // line of windows at a time.
  constexpr int32_t kLine = 16;
  const int64_t lines = (nwin + kLine - 1) / kLine;
  RawArray<uint32_t> wrel(nb * nwin);
  std::vector<int32_t> wlen(nwin, 0);
  std::vector<int64_t> wseg(nwin + 1, 0);
  parallel_dynamic(lines, nt, 1, [&](int64_t l) {
    const int32_t w0 = static_cast<int32_t>(l) * kLine, w1 = std::min(nwin, w0 + kLine);
    uint32_t run[kLine] = {};
    int32_t segs[kLine] = {};
    for (int64_t b = 0; b < nb; b++) {
      const uint32_t* o = &boff[b * pitch];
      uint32_t* r = &wrel[b * nwin];
      for (int32_t w = w0; w < w1; w++) {
        const uint32_t d = o[w + 1] - o[w];
        r[w] = run[w - w0];
        run[w - w0] += d;
        segs[w - w0] += d > 0;
      }
    }
    for (int32_t w = w0; w < w1; w++) {
      wlen[w] = static_cast<int32_t>(run[w - w0]);
      wseg[w + 1] = segs[w - w0];
    }
  });
  std::vector<int64_t> wstart(nwin + 1, 0), wgroup(nwin + 1, 0);  // window starts padded
  for (int32_t w = 0; w < nwin; w++) {
    wstart[w + 1] = wstart[w] + (int64_t(wlen[w]) + kBPer - 1) / kBPer * kBPer;
    wgroup[w + 1] = wgroup[w] + (wlen[w] + 63) / 64;
    wseg[w + 1] += wseg[w];
  }
  // 4. Segment tables per window (non-empty segments, bucket order), and where
  // segments start, per group of 64 edges.
  RawArray<int32_t> seg_e(wseg[nwin]), seg_d(wseg[nwin]);
  parallel_dynamic(lines, nt, 1, [&](int64_t l) {
    const int32_t w0 = static_cast<int32_t>(l) * kLine, w1 = std::min(nwin, w0 + kLine);
    int64_t at[kLine];
    for (int32_t w = w0; w < w1; w++) at[w - w0] = wseg[w];
    for (int64_t b = 0; b < nb; b++) {
      const uint32_t* o = &boff[b * pitch];
      const uint32_t* r = &wrel[b * nwin];
      for (int32_t w = w0; w < w1; w++) {
        if (o[w + 1] == o[w]) continue;
        const int64_t k = at[w - w0]++;
        seg_e[k] = static_cast<int32_t>(r[w]);
        seg_d[k] = static_cast<int32_t>(bstart[b] + o[w] - r[w]);
      }
    }
  });
  RawArray<BlockGroup> groups(wgroup[nwin]);
  parallel_dynamic(nwin, nt, 1, [&](int64_t w) {
    int32_t k = 0;
    const int32_t* se = seg_e.data() + wseg[w];
    const int32_t ns = static_cast<int32_t>(wseg[w + 1] - wseg[w]);
    for (int64_t g = wgroup[w]; g < wgroup[w + 1]; g++) {
      const int32_t e0 = static_cast<int32_t>(g - wgroup[w]) * 64;
      while (k + 1 < ns && se[k + 1] <= e0) k++;
      groups[g] = {0, k, 0};
      for (int32_t j = k + 1; j < ns && se[j] < e0 + 64; j++) groups[g].starts |= uint64_t(1) << (se[j] - e0 - 1);
    }
  });
  // 5. Fine buckets: rows by length, longest first (row order inside a length
  // class of powers of two, so that the rows of a wavefront are alike), and
  // their runs of places in that order.
  RawArray<FineRow> rows(shape.fine ? n : 0);
  RawArray<int32_t> place(shape.fine ? n : 0);  // each row's next place
  std::vector<int32_t> nlong(nb, 0), nmid(nb, 0);
  if (shape.fine)
    parallel_dynamic(nb, nt, 16, [&](int64_t b) {
      if (brow[b + 1] - brow[b] == 1) {  // one-row units need no order
        rows[brow[b]] = {};
        return;
      }
      auto len = [&](int64_t r) { return off[r + 1] - off[r]; };
      auto cls = [&](int64_t r) {  // 0: longest, 64: empty
        return len(r) == 0 ? 64 : __builtin_clzll(static_cast<unsigned long long>(len(r)));
      };
      int64_t at[66] = {};
      for (int64_t r = brow[b]; r < brow[b + 1]; r++) {
        at[cls(r) + 1]++;
        nlong[b] += len(r) >= kFineLong;
        nmid[b] += len(r) >= kFineMid && len(r) < kFineLong;
      }
      for (int c = 0; c < 65; c++) at[c + 1] += at[c];
      for (int64_t r = brow[b]; r < brow[b + 1]; r++)
        rows[brow[b] + at[cls(r)]++] = {static_cast<uint16_t>(r - brow[b]), 0, static_cast<uint16_t>(len(r)), 0};
      int32_t next = 0;
      for (int64_t i = brow[b]; i < brow[b + 1]; i++) {
        rows[i].start = static_cast<uint16_t>(next);
        place[brow[b] + rows[i].row] = next;
        next += rows[i].len;
      }
    });
  // 6. Fill both arrays, bucket by bucket (disjoint segments); the tables' words
  // are each segment's next place in them.
  RawArray<uint16_t> src(std::max<int64_t>(1, wstart[nwin]));
  RawArray<uint16_t> brow_off(std::max<int64_t>(1, m));
  src[0] = brow_off[0] = 0;
  for (int32_t w = 0; w < nwin; w++) std::fill(&src[0] + wstart[w] + wlen[w], &src[0] + wstart[w + 1], uint16_t(0));
  parallel_dynamic(nb, nt, 4, [&](int64_t b) {
    const bool places = shape.fine && brow[b + 1] - brow[b] > 1;
    uint32_t* o = &boff[b * pitch];
    uint32_t* p = &wrel[b * nwin];
    uint16_t* const to = &brow_off[0] + bstart[b];
    for (int64_t r = brow[b]; r < brow[b + 1]; r++)
      for (int64_t e = off[r]; e < off[r + 1]; e++) {
        const uint32_t w = window(nbr[e]);
        src[wstart[w] + p[w]++] = static_cast<uint16_t>(static_cast<uint32_t>(nbr[e]) % kBWin);
        to[o[w]++] = static_cast<uint16_t>(places ? place[r]++ : r - brow[b]);
      }
  });
  // 7. Units: a bucket whole, or a one-row bucket beyond shape.edges in parts
  // whose sums go to partial slots.
  std::vector<BlockUnit> units;
  std::vector<BlockSplit> splits;
  int32_t slots = 0;
  for (int64_t b = 0; b < nb; b++) {
    const int64_t e0 = bstart[b], e1 = bstart[b + 1];
    if (e1 - e0 <= shape.edges) {
      units.push_back({brow[b], brow[b + 1] - brow[b], -1, nlong[b], nmid[b], 0, e0, e1});
      continue;
    }
    const int32_t first = slots;
    for (int64_t e = e0; e < e1; e += shape.edges)
      units.push_back({brow[b], 1, slots++, 0, 0, 0, e, std::min(e1, e + shape.edges)});
    splits.push_back({brow[b], first, slots - first, 0});
  }
  out->src.swap(src);
  out->wstart.swap(wstart);
  out->wlen.swap(wlen);
  out->wseg.swap(wseg);
  out->seg_e.swap(seg_e);
  out->seg_d.swap(seg_d);
  out->wgroup.swap(wgroup);
  out->groups.swap(groups);
  out->brow_off.swap(brow_off);
  out->rows.swap(rows);
  out->units.swap(units);
  out->splits.swap(splits);
  out->n_slots = slots;
  out->n_windows = nwin;
  out->n_buckets = nb;
  return DMM_OK;
}

namespace {

template <typename Array>
int upload_vec(dmm_ctx* ctx, void** dst, const Array& v, const char* what) {
  const size_t bytes = sizeof(*v.data()) * v.size();
  int rc = dev_alloc(ctx, dst, std::max(sizeof(*v.data()), bytes), what);
  if (rc) return rc;
  if (bytes) DMM_HIP_CHECK(ctx, hipMemcpy(*dst, v.data(), bytes, hipMemcpyHostToDevice));
  return DMM_OK;
}

}  // namespace

// Fine buckets of a block with m in-edges: as large as LDS allows, in a small
// block so that every workgroup (two per CU) has one.  Larger blocks gain
// nothing from smaller buckets that would divide evenly: Kronecker-23, block
// 3 of 8 (33 M edges, 4.5 full buckets per workgroup): pass 2 75 us, 90 us
// with buckets of 13900 edges.
BlockShape fine_shape(int64_t m, int cus) {
  BlockShape shape = kFine;
  const int64_t groups = 2 * std::max(1, cus);
  shape.edges = std::min<int64_t>(kFineEdges, std::max<int64_t>(kFineLeast, ceil_div(m, groups)));
  return shape;
}

// Whether a block's iteration is faster with the fine buckets of fine_shape
// than with coarse ones, from what the two shapes take beyond what they have in
// common (us; each term fitted to blocks of 2 to 126 M edges from 2^23 to 2^27
// sources):
//   fine    3.5 per M edges (both passes), 13 per M segments: pass 1 writes a
//           segment at a time, and the more windows, the shorter they are
//   coarse  1.6 per M edges (pass 1), 13 per M segments (few), and the edges of
//           the workgroup that has most (pass 2): 0.42 ns for each, and 0.37
//           for one that follows another of its row in a segment, whose LDS
//           atomics wait for each other; 0.1 ns for those of one-row units
// So blocks of like rows are better coarse from some 50 M edges on, or 30 M from
// many windows (uniform, 2^23 sources, 67 M: fine 272 us, coarse 225; 2^25, 126
// M: 645, 467; 2^27, 34 M: 321, 286; 2^25, 34 M: 179, 198), Kronecker blocks,
// whose hubs crowd one coarse unit, only where the fine buckets hardly fit
// (Kronecker-24, an eighth, 66 M: 321, 437; -26, a 32nd: 452, 548; -25, a ninth,
// 117 M: 648, 641).  Of 60 blocks measured both ways none was 5% slower than
// the better.
constexpr double kFineEdgeUs = 3.5e-6, kCoarseEdgeUs = 1.6e-6, kSegmentUs = 13e-6;
constexpr double kAtomicUs = 0.42e-3, kRepeatUs = 0.37e-3, kOneRowUs = 0.1e-3;

bool fine_is_faster(int64_t n, int64_t n_gather, const int64_t* off, const int32_t* nbr, int cus, double* us) {
  const double m = static_cast<double>(off[n]);
  const double nwin = static_cast<double>(std::max<int64_t>(1, ceil_div(n_gather, kBWin)));
  const BlockShape fine = fine_shape(off[n], cus);
  const double nb_fine = static_cast<double>(cut_buckets(n, off, fine).size()) - 1;
  us[0] = kFineEdgeUs * m;
  us[1] = kCoarseEdgeUs * m;
  if (nb_fine > kBSegMax) return false;
  const std::vector<int32_t> coarse = cut_buckets(n, off, kCoarse);
  const int64_t nb_coarse = static_cast<int64_t>(coarse.size()) - 1;
  // Pass 2 of the coarse units, dealt in turn.
  std::vector<double> load(std::max(1, cus), 0.0);
  size_t unit = 0;
  for (int64_t b = 0; b < nb_coarse; b++) {
    const int64_t edges = off[coarse[b + 1]] - off[coarse[b]];
    if (coarse[b + 1] - coarse[b] == 1) {
      for (int64_t e = 0; e < std::max<int64_t>(1, edges); e += kCoarse.edges)
        load[unit++ % load.size()] += kOneRowUs * static_cast<double>(std::min(kCoarse.edges, edges - e));
      continue;
    }
    double repeats = 0;
    for (int64_t r = coarse[b]; r < coarse[b + 1]; r++) {
      const double d = static_cast<double>(off[r + 1] - off[r]);
      // Edges less the segments that they fall into.
      if (d > 1) repeats += d - nwin * -std::expm1(-d / nwin);
    }
    load[unit++ % load.size()] += kAtomicUs * static_cast<double>(edges) + kRepeatUs * std::max(0.0, repeats);
  }
  us[1] += *std::max_element(load.begin(), load.end());
  // At most a segment per edge, and per window and bucket.
  if (us[0] + kSegmentUs * std::min(m, nb_fine * nwin) <= us[1]) return true;
  if (us[0] > us[1] + kSegmentUs * std::min(m, static_cast<double>(nb_coarse) * nwin)) return false;
  // Else those of buckets of the same size: a window that has the share p of
  // the edges is met by 1 - (1 - p)^(edges) of them.
  const int nt = resolve_threads(0);
  std::vector<std::vector<uint32_t>> part(nt, std::vector<uint32_t>(static_cast<size_t>(nwin), 0));
  parallel_dynamic(nt, nt, 1, [&](int64_t t) {
    std::vector<uint32_t>& c = part[t];
    for (int64_t e = off[n] * t / nt; e < off[n] * (t + 1) / nt; e++) c[static_cast<uint32_t>(nbr[e]) / kBWin]++;
  });
  double segs_fine = 0, segs_coarse = 0;
  for (size_t w = 0; w < static_cast<size_t>(nwin); w++) {
    double p = 0;
    for (const auto& c : part) p += c[w];
    p /= m;
    segs_fine += nb_fine * -std::expm1(-m / nb_fine * p);
    segs_coarse += static_cast<double>(nb_coarse) * -std::expm1(-m / static_cast<double>(nb_coarse) * p);
  }
  us[0] += kSegmentUs * segs_fine;
  us[1] += kSegmentUs * segs_coarse;
  return us[0] <= us[1];
}

int pr_blocks_build(dmm_ctx* ctx) {
  const int64_t n = ctx->nloc;
  const int64_t m = ctx->m_in;
  RawArray<int64_t> off(n + 1);
  RawArray<int32_t> nbr(std::max<int64_t>(1, m));
  DMM_HIP_CHECK(ctx, hipMemcpy(off.data(), ctx->d_in_off, sizeof(int64_t) * (n + 1), hipMemcpyDeviceToHost));
  if (m > 0) DMM_HIP_CHECK(ctx, hipMemcpy(nbr.data(), ctx->d_in_nbr, sizeof(int32_t) * m, hipMemcpyDeviceToHost));
  BlockHost bh;
  std::string err;
  const int64_t held = ctx->dev_bytes;
  double us[2];
  ctx->bp_fine = m < (int64_t(1) << 31) && fine_is_faster(n, ctx->n, off.data(), nbr.data(), ctx->cu_count, us);
  int rc = build_blocks_host(n, ctx->n, off.data(), nbr.data(), ctx->bp_fine ? fine_shape(m, ctx->cu_count) : kCoarse,
                             &bh, &err);
  if (rc) return set_err(ctx, rc, "%s", err.c_str());
  RawArray<int64_t>().swap(off);
  RawArray<int32_t>().swap(nbr);
  if ((rc = upload_vec(ctx, &ctx->d_bp_src, bh.src, "PR block sources")) ||
      (rc = upload_vec(ctx, &ctx->d_bp_wstart, bh.wstart, "PR block window starts")) ||
      (rc = upload_vec(ctx, &ctx->d_bp_wlen, bh.wlen, "PR block window lengths")) ||
      (rc = upload_vec(ctx, &ctx->d_bp_wseg, bh.wseg, "PR block window segments")) ||
      (rc = upload_vec(ctx, &ctx->d_bp_wgroup, bh.wgroup, "PR block groups")) ||
      (rc = upload_vec(ctx, &ctx->d_bp_groups, bh.groups, "PR block groups")) ||
      (rc = upload_vec(ctx, &ctx->d_bp_seg_d, bh.seg_d, "PR block segment destinations")) ||
      (rc = upload_vec(ctx, &ctx->d_bp_brow, bh.brow_off, "PR block row offsets")) ||
      (rc = upload_vec(ctx, &ctx->d_bp_rows, bh.rows, "PR block rows")) ||
      (rc = upload_vec(ctx, &ctx->d_bp_units, bh.units, "PR block units")) ||
      (rc = upload_vec(ctx, &ctx->d_bp_splits, bh.splits, "PR block split rows")) ||
      // One spare slot past the m contributions takes the propagation
      // pass's stores from lanes past a window's end.
      (rc = dev_alloc(ctx, &ctx->d_bp_val, sizeof(float) * (m + 1), "PR block contributions")) ||
      (rc = dev_alloc(ctx, &ctx->d_bp_part, 16 * std::max<int64_t>(1, bh.n_slots), "PR block split partials"))) {
    ctx->bp_bytes = ctx->dev_bytes - held;  // what the failed build holds, freed with the layout
    return rc;
  }
  ctx->n_bp_windows = bh.n_windows;
  ctx->n_bp_units = static_cast<int64_t>(bh.units.size());
  ctx->n_bp_splits = static_cast<int64_t>(bh.splits.size());
  ctx->n_bp_buckets = bh.n_buckets;
  ctx->bp_bytes = ctx->dev_bytes - held;
  ctx->bp_ready = true;
  return DMM_OK;
}

namespace {

constexpr int kHostFxShift = 80;  // as the device's kFxShift

// Host restatement of the device's fx_of: c * 2^80 as a 128-bit two's
// complement integer, truncated below 2^-80.
__int128 host_fx_of(float c) {
  uint32_t bits;
  std::memcpy(&bits, &c, 4);
  const int e = static_cast<int>((bits >> 23) & 0xFFu);
  const unsigned __int128 m = (bits & 0x7FFFFFu) | 0x800000u;
  if (e == 0) return 0;
  const int sh = e - 150 + kHostFxShift;
  if (sh <= -24) return 0;
  const unsigned __int128 x = sh < 0 ? m >> (-sh) : m << sh;
  return (bits >> 31) ? -static_cast<__int128>(x) : static_cast<__int128>(x);
}

// Host restatement of fx_value: the top 64 significant bits with a sticky
// bit, one rounding to FP32, then the exact power-of-two scaling.
float host_fx_value(__int128 v) {
  const bool neg = v < 0;
  const unsigned __int128 a = neg ? static_cast<unsigned __int128>(-v) : static_cast<unsigned __int128>(v);
  const uint64_t hi = static_cast<uint64_t>(a >> 64), lo = static_cast<uint64_t>(a);
  float f;
  if (hi == 0) {
    f = std::ldexp(static_cast<float>(lo), -kHostFxShift);
  } else {
    const int lz = __builtin_clzll(hi);
    const uint64_t top = lz ? (hi << lz) | (lo >> (64 - lz)) : hi;
    const uint64_t rest = lz ? lo << lz : lo;
    f = std::ldexp(static_cast<float>(top | (rest != 0 ? 1ull : 0ull)), 64 - lz - kHostFxShift);
  }
  return neg ? -f : f;
}

// Checks every index the kernels use against its buffer and that every edge
// reaches its row once, and replays pass 1 and pass 2 with the kernels'
// arithmetic.
int check_blocks(const BlockHost& bh, const BlockShape& shape, int64_t n, int64_t n_gather, const int64_t* off,
                 const float* contrib, float* incoming) {
  const int64_t m = off[n];
  auto bad = [](const char* what) { return set_err(nullptr, DMM_ERR_GRAPH, "block layout: %s", what); };
  const int32_t nwin = bh.n_windows;
  if (static_cast<int32_t>(bh.wstart.size()) != nwin + 1 || static_cast<int32_t>(bh.wseg.size()) != nwin + 1 ||
      static_cast<int64_t>(bh.brow_off.size()) < std::max<int64_t>(1, m) || bh.n_buckets > kBSegMax)
    return bad("sizes");
  // Pass 1, window by window, as k_bprop walks it.
  std::vector<float> val(std::max<int64_t>(1, m), 0.0f);
  std::vector<char> hit(std::max<int64_t>(1, m), 0);
  for (int32_t w = 0; w < nwin; w++) {
    const int64_t base = int64_t(w) * kBWin;
    const int64_t cnt = std::min<int64_t>(kBWin, n_gather - base);
    const int64_t s0 = bh.wseg[w];
    const int ns = static_cast<int>(bh.wseg[w + 1] - s0);
    const int len = bh.wlen[w];
    if (ns < 0 || ns > kBSegMax || bh.wstart[w] % kBPer || bh.wstart[w] + len > bh.wstart[w + 1]) return bad("window");
    if (ns > 0 && bh.seg_e[s0] != 0) return bad("first segment");
    for (int k = 1; k < ns; k++)
      if (bh.seg_e[s0 + k] <= bh.seg_e[s0 + k - 1] || bh.seg_e[s0 + k] >= len) return bad("segment starts");
    if (bh.wgroup[w + 1] - bh.wgroup[w] != (len + 63) / 64) return bad("groups");
    for (int i = 0; i < len; i++) {
      const BlockGroup& g = bh.groups[bh.wgroup[w] + i / 64];
      const int k = i % 64;
      const int sg = g.first + __builtin_popcountll(k ? g.starts << (64 - k) : 0);
      if (sg < 0 || sg >= ns || bh.seg_e[s0 + sg] > i || (sg + 1 < ns && bh.seg_e[s0 + sg + 1] <= i))
        return bad("group segments");
      const int64_t dst = int64_t(bh.seg_d[s0 + sg]) + i;
      const uint16_t s = bh.src[bh.wstart[w] + i];
      if (s >= cnt) return bad("source offset");
      if (dst < 0 || dst >= m || hit[dst]) return bad("destination");
      hit[dst] = 1;
      val[dst] = contrib[base + s];
    }
  }
  for (int64_t e = 0; e < m; e++)
    if (!hit[e]) return bad("destination never written");
  // Pass 2, unit by unit, and the split rows; every row finishes once and
  // every unit holds exactly its rows' in-edges.
  std::vector<__int128> part(std::max(1, bh.n_slots), 0);
  std::vector<int64_t> slot_edges(std::max(1, bh.n_slots), 0);
  std::vector<char> done(std::max<int64_t>(1, n), 0);
  int64_t next_e = 0;
  for (const BlockUnit& u : bh.units) {
    if (u.e0 != next_e || u.e1 < u.e0 || u.nrows < 1 || u.nrows > shape.rows || u.e1 - u.e0 > shape.edges ||
        u.row0 < 0 || int64_t(u.row0) + u.nrows > n)
      return bad("unit");
    next_e = u.e1;
    if (u.slot >= 0) {
      if (u.nrows != 1 || u.slot >= bh.n_slots) return bad("split unit");
      __int128 s = 0;
      for (int64_t e = u.e0; e < u.e1; e++) {
        if (!shape.fine && bh.brow_off[e] != 0) return bad("split unit row");
        s += host_fx_of(val[e]);
      }
      part[u.slot] = s;
      slot_edges[u.slot] = u.e1 - u.e0;
      continue;
    }
    if (off[u.row0 + u.nrows] - off[u.row0] != u.e1 - u.e0) return bad("unit edges differ from its rows' in-edges");
    std::vector<__int128> acc(u.nrows, 0);
    if (shape.fine && u.nrows > 1) {
      // As k_bfine: every contribution to its place, then each row's run.
      if (u.nlong > kFineEdges / kFineLong) return bad("long rows");
      std::vector<float> place(u.e1 - u.e0);
      std::vector<char> set(u.e1 - u.e0, 0);
      for (int64_t e = u.e0; e < u.e1; e++) {
        const int64_t at = bh.brow_off[e];
        if (at >= u.e1 - u.e0 || set[at]) return bad("place in row order");
        set[at] = 1;
        place[at] = val[e];
      }
      std::vector<char> taken(u.nrows, 0);
      int64_t next_place = 0;
      for (int32_t i = 0; i < u.nrows; i++) {
        const FineRow fr = bh.rows[u.row0 + i];
        const int32_t r = fr.row;
        if (r >= u.nrows || taken[r]) return bad("row order");
        taken[r] = 1;
        const int64_t s = next_place, e = s + (off[u.row0 + r + 1] - off[u.row0 + r]);
        if (fr.start != s || fr.len != e - s) return bad("row places");
        next_place = e;
        if ((e - s >= kFineLong) != (i < u.nlong) || (e - s >= kFineMid) != (i < u.nlong + u.nmid))
          return bad("row classes");
        for (int64_t k = s; k < e; k++) acc[r] += host_fx_of(place[k]);
      }
    } else {
      for (int64_t e = u.e0; e < u.e1; e++) {
        if (bh.brow_off[e] >= u.nrows) return bad("row offset");
        acc[bh.brow_off[e]] += host_fx_of(val[e]);
      }
    }
    for (int32_t r = 0; r < u.nrows; r++) {
      incoming[u.row0 + r] = host_fx_value(acc[r]);
      done[u.row0 + r]++;
    }
  }
  if (next_e != m) return bad("units do not cover the edges");
  for (const BlockSplit& sp : bh.splits) {
    if (sp.row < 0 || sp.row >= n || sp.first < 0 || sp.count < 1 || sp.first + sp.count > bh.n_slots)
      return bad("split row");
    __int128 s = 0;
    int64_t edges = 0;
    for (int j = 0; j < sp.count; j++) {
      s += part[sp.first + j];
      edges += slot_edges[sp.first + j];
    }
    if (edges != off[sp.row + 1] - off[sp.row]) return bad("split row edges");
    incoming[sp.row] = host_fx_value(s);
    done[sp.row]++;
  }
  for (int64_t r = 0; r < n; r++)
    if (done[r] != 1) return bad("row not finished exactly once");
  return DMM_OK;
}

}  // namespace

}  // namespace dmm

// Host check of the PE-block propagation layout (no GPU): the coarse layout,
// and fine ones where the block has them, whose sums must be the same.
extern "C" int dmm_pr_blocks_check(int64_t n, int64_t n_gather, const int64_t* off, const int32_t* nbr,
                                   const float* contrib, float* incoming, int64_t* stats) {
  using namespace dmm;
  if (n < 0 || !off || (off[n] > 0 && !nbr) || !contrib || !incoming || !stats)
    return set_err(nullptr, DMM_ERR_INVALID, "dmm_pr_blocks_check: bad arguments");
  for (int64_t e = 0; e < off[n]; e++)
    if (nbr[e] < 0 || nbr[e] >= n_gather) return set_err(nullptr, DMM_ERR_GRAPH, "source outside [0, n_gather)");
  BlockHost bh;
  std::string err;
  int rc = build_blocks_host(n, n_gather, off, nbr, kCoarse, &bh, &err);
  if (rc) return set_err(nullptr, rc, "%s", err.c_str());
  if ((rc = check_blocks(bh, kCoarse, n, n_gather, off, contrib, incoming))) return rc;
  // The largest and the smallest fine buckets the GPU uses.
  BlockShape least = kFine;
  least.edges = kFineLeast;
  for (const BlockShape& shape : {kFine, least}) {
    BlockHost fine;
    rc = build_blocks_host(n, n_gather, off, nbr, shape, &fine, &err);
    if (rc == DMM_ERR_CAPACITY) continue;
    if (rc) return set_err(nullptr, rc, "%s", err.c_str());
    std::vector<float> again(std::max<int64_t>(1, n), 0.0f);
    if ((rc = check_blocks(fine, shape, n, n_gather, off, contrib, again.data()))) return rc;
    if (n > 0 && std::memcmp(again.data(), incoming, sizeof(float) * n) != 0)
      return set_err(nullptr, DMM_ERR_GRAPH, "block layout: fine and coarse sums differ");
  }
  stats[0] = bh.n_windows;
  stats[1] = bh.n_buckets;
  stats[2] = static_cast<int64_t>(bh.units.size());
  stats[3] = static_cast<int64_t>(bh.splits.size());
  stats[4] = static_cast<int64_t>(bh.seg_e.size());
  stats[5] = bh.n_slots;
  return DMM_OK;
}

// Host check of the choice between the shapes: 1 if a block's iteration on a
// GPU of `cus` CUs would take fine buckets; us[2]: the estimates that decided
// it, as far as they were needed.
extern "C" int dmm_pr_blocks_shape(int64_t n, int64_t n_gather, const int64_t* off, const int32_t* nbr, int32_t cus,
                                   double* us) {
  using namespace dmm;
  if (n < 0 || !off || (off[n] > 0 && !nbr) || !us || cus < 1)
    return set_err(nullptr, DMM_ERR_INVALID, "dmm_pr_blocks_shape: bad arguments");
  for (int64_t e = 0; e < off[n]; e++)
    if (nbr[e] < 0 || nbr[e] >= n_gather) return set_err(nullptr, DMM_ERR_GRAPH, "source outside [0, n_gather)");
  return fine_is_faster(n, n_gather, off, nbr, cus, us) ? 1 : 0;
}
