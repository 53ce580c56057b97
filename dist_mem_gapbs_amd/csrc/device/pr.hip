// Pull-direction PageRank on gfx950.
//
// Reference: PageRankPull, src/pr.cc:41-70 (oracle gapbs-verify/pr.cc:34-59):
//   contrib[v] = score[v] / out_degree(v)
//   score[u]   = (1 - d)/N + d * sum_{v in in(u)} contrib[v]      (d = 0.85f)
//   error      = sum_u |score_new[u] - score_old[u]|  (double), stop < eps.
// Data in HBM: in-CSR (int64 offsets, int32 IDs), score[nloc], contrib in two
// buffers (the iteration reads one and writes the next), per-block error
// partials and a small control block.  Each iteration is one pass over the
// CSR: the kernel that finishes vertex u's sum also writes its new score and
// its next contribution, so an iteration moves 8M + 20N bytes (FP32).
//
// Three arithmetic modes:
//   FP32_SERIAL  the reference's arithmetic exactly: FP32 sums in ascending
//                in-neighbour order (thread per light row, lane per bundled
//                row, exact composition of the additions in long rows).
//   FP32_KAHAN   FP32 storage and gathers, each sum compensated (Knuth's
//                TwoSum error-free transformation, TAOCP Vol. 2 4.2.2;
//                partial (sum, error) pairs merged with TwoSum as in
//                Ogita-Rump-Oishi Sum2).  Result within ~1 ulp of the exact
//                sum plus O(n u^2) -- far below the FP32 score rounding.
//   FP64         FP64 scores, contributions and sums.
// The L1 error is accumulated in FP64 per block and reduced in a fixed
// order, so every mode is run-to-run deterministic.
#include "pr.h"

#include <algorithm>
#include <mutex>

#include "layout.h"

namespace dmm {

namespace {

constexpr int kThreads = 256;
constexpr int kGroup = 4;         // lanes per light vertex (KAHAN / FP64)
constexpr int kUnroll = 8;        // gathers in flight per lane on heavy items
constexpr int kTailUnroll = 4;    // ... on what they leave
constexpr int kLightUnroll = 4;   // gathers in flight per lane on light rows
constexpr int kFusedThreads = 1024;
constexpr int kHubBytes = 128 * 1024;  // LDS copy of the first contributions

struct PrParams {
  double eps;
  float base_f, damp_f;           // (1 - 0.85f) / N, 0.85f
  double base_d, damp_d;          // widened FP32 constants for FP64 mode
  float init_f;
  float pad;
  double init_d;
};

struct PrArgs {
  const int64_t* in_off;          // local rows
  const int32_t* in_nbr;          // global IDs
  const int64_t* out_off;         // local rows (out-degree for contrib)
  const int32_t* heavy;           // local rows with in-degree >= heavy_threshold, longest class first
  const PrItem* items;            // heavy rows / segments of split rows
  const PrSuper* supers;          // split rows and their segment slots
  double2* partial;               // per-segment partial sums
  int64_t nloc, n_heavy, n_items, n_super;
  const SerialItem* sitems;       // serial mode: each workgroup's items
  const int32_t* sstart;          // ... first item of each workgroup (+ end)
  int64_t n_gather;               // entries of the gathered contribution vector
  int64_t light_begin, light_end; // light-row range (heavy rows inside are skipped)
  int64_t zero_begin;             // rows [zero_begin, nloc) have no in-edges
  int heavy_threshold;
  double* err_part;               // [main | super] blocks
  int serial_hub;                     // contributions [0, serial_hub) go to LDS (serial mode)
  int super_blocks;
  int main_blocks;                // error partials written before the combine
  PrCtrl* ctrl;
  double* err_trace;              // per-iteration error
  double* err_out;                // the iteration's error again, for the caller (may be NULL)
  const PrParams* prm;
};

// What an iteration's first kernel needs of the iteration before.
struct PrPrev {
  const double* part;   // its error partials
  int parts;
  int it;               // this iteration's number: 0 has none before it
  PrCtrl* ctrl;
  double* err_trace;
  const PrParams* prm;
};

// Constants and control block of a block iteration, written by its first
// kernel, where they are not there yet (prm NULL: they are).
struct PrHead {
  PrParams* prm;
  PrCtrl* ctrl;
  PrParams p;
};

__device__ __forceinline__ void write_head(const PrHead& h) {
  *h.prm = h.p;
  h.ctrl->err = 0;
  h.ctrl->ticket = 0;
  h.ctrl->pad = 0;
}

__global__ void k_head(PrHead h) {
  if (blockIdx.x == 0 && threadIdx.x == 0) write_head(h);
}

// The sum of an iteration's error partials by a workgroup of kBlock threads,
// in one order whoever takes it: what a run reports, and where it stops, must
// not depend on which kernel of which captured chain sums an iteration.  The
// order is that of the kThreads threads of k_reduce; the others of a larger
// workgroup add nothing.  Partial `own` (-1: none) is `mine`.  The sum is every
// thread's; scratch (one double per wavefront) is in use until the next barrier.
template <int kBlock>
__device__ __forceinline__ double error_sum(const double* part, int parts, int own, double mine, double* scratch) {
  double x = 0;
  if (threadIdx.x < kThreads)
    for (int i = threadIdx.x; i < parts; i += kThreads) x += i == own ? mine : part[i];
  x = wave_sum(x);
  if (lane_id() == 0) scratch[threadIdx.x >> 6] = x;
  __syncthreads();
  double t = 0;
  for (int w = 0; w < kThreads / 64; w++) t += scratch[w];
  return t;
}

// Start of an iteration's first kernel: every workgroup sums the previous
// iteration's error partials in the same order and stops if that iteration
// converged (src/pr.cc:66-68); workgroup 0 records the error and the stop
// decision for the kernels that follow.  ctrl->ticket counts the iterations
// run; ctrl->pad != 0 marks convergence and turns the remaining captured
// iterations into no-ops.  A kernel of its own for this took 5 us an
// iteration.  scratch: kBlock / 64 + 1 doubles of LDS, free again on return.
template <int kBlock>
__device__ __forceinline__ bool pr_begin(const PrPrev& p, double* scratch) {
  if (p.it == 0) return true;
  // Workgroup 0 may be writing the mark: one thread reads it for all.
  if (threadIdx.x == 0) scratch[kBlock / 64] = p.ctrl->pad ? 1.0 : 0.0;
  const double t = error_sum<kBlock>(p.part, p.parts, -1, 0.0, scratch);
  const bool over = scratch[kBlock / 64] != 0.0;
  __syncthreads();
  if (over) return false;
  const bool converged = t < p.prm->eps;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    p.ctrl->err = t;
    p.ctrl->ticket = p.it;
    if (p.it <= DMM_MAX_PR_ITERS) p.err_trace[p.it - 1] = t;
    if (converged) p.ctrl->pad = 1;
  }
  return !converged;
}

__device__ __forceinline__ void two_sum(float a, float b, float& s, float& e) {
  s = a + b;
  const float bb = s - a;
  e = (a - (s - bb)) + (b - bb);
}

struct Comp {
  float s, c;
  __device__ __forceinline__ void add(float x) {
    float t, e;
    two_sum(s, x, t, e);
    s = t;
    c += e;
  }
  __device__ __forceinline__ void merge(float s2, float c2) {
    float t, e;
    two_sum(s, s2, t, e);
    s = t;
    c = (c + c2) + e;
  }
  __device__ __forceinline__ float value() const { return s + c; }
};

template <int kBlock = kThreads>
__device__ __forceinline__ double block_err_sum(double x, double* red) {
  double s = wave_sum(x);
  if (lane_id() == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  double r = 0;
  if (threadIdx.x == 0)
    for (int w = 0; w < kBlock / 64; w++) r += red[w];
  __syncthreads();
  return r;
}

__device__ __forceinline__ int64_t out_deg(const PrArgs& a, int64_t lu) {
  return a.out_off[lu + 1] - a.out_off[lu];
}

// Finishes vertex lu given its incoming sum: new score, next contribution
// and the |delta| term (src/pr.cc:61-63, 52-53).
__device__ __forceinline__ double finish_f32(const PrArgs& a, int64_t lu, float incoming,
                                             float* score, float* contrib_out) {
  const float old_score = score[lu];
  const float nw = a.prm->base_f + a.prm->damp_f * incoming;
  score[lu] = nw;
  contrib_out[lu] = nw / static_cast<float>(out_deg(a, lu));
  return static_cast<double>(fabsf(nw - old_score));
}

__device__ __forceinline__ double finish_f64(const PrArgs& a, int64_t lu, double incoming,
                                             double* score, double* contrib_out) {
  const double old_score = score[lu];
  const double nw = a.prm->base_d + a.prm->damp_d * incoming;
  score[lu] = nw;
  contrib_out[lu] = nw / static_cast<double>(out_deg(a, lu));
  return fabs(nw - old_score);
}

// Inclusive prefix sum over the 64 lanes from DPP lane moves (row_shr
// 1/2/4/8 inside 16-lane rows, row_bcast 15 and 31 across): no LDS traffic.
__device__ __forceinline__ uint32_t wave_scan_u32(uint32_t v) {
  v += __builtin_amdgcn_update_dpp(0u, v, 0x111, 0xf, 0xf, true);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0u, v, 0x112, 0xf, 0xf, true);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0u, v, 0x114, 0xf, 0xf, true);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0u, v, 0x118, 0xf, 0xf, true);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0u, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0u, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return v;
}

// Block-wide copy of cnt entries from src into LDS (room for kBytes, a
// multiple of 16) with all 16-byte loads of a thread issued before its
// stores (one round trip instead of one per element): whole when cnt fills
// the room, else the loads past the last whole one repeat it and a tail
// follows.  A src that is not 16-byte aligned is copied entry by entry.
template <typename T, int kBytes, int kBlock = kFusedThreads>
__device__ __forceinline__ void lds_fill(T* dst, const T* __restrict__ src, int cnt) {
  constexpr int kPer = kBytes / 16 / kBlock;
  constexpr int kVec = 16 / sizeof(T);
  static_assert(kBytes % (16 * kBlock) == 0, "fill size");
  const int n4 = (reinterpret_cast<uintptr_t>(src) & 15) == 0 ? cnt / kVec : 0;
  if (n4 > 0) {
    float4 v[kPer];
#pragma unroll
    for (int i = 0; i < kPer; i++)
      v[i] = reinterpret_cast<const float4*>(src)[min(static_cast<int>(threadIdx.x) + i * kBlock, n4 - 1)];
#pragma unroll
    for (int i = 0; i < kPer; i++)
      if (static_cast<int>(threadIdx.x) + i * kBlock < n4) reinterpret_cast<float4*>(dst)[threadIdx.x + i * kBlock] = v[i];
  }
  for (int j = n4 * kVec + threadIdx.x; j < cnt; j += kBlock) dst[j] = src[j];
}

// The contributions of the vertices u[j], j-th edge at k + j * stride of those
// below e (past it +0, which changes no sum here: they start at +0).  Every
// lane loads from both the hub and HBM, where the other has the vertex the
// first entry, and selects when both are there: with a branch, either load of
// an edge waited for the other of the edge before.
template <typename T, int kN>
__device__ __forceinline__ void hub_gathers(const T* hub, int hub_n, const T* __restrict__ cin,
                                            const int32_t (&u)[kN], int64_t k, int stride, int64_t e, T (&x)[kN]) {
  T far[kN], near[kN];
#pragma unroll
  for (int j = 0; j < kN; j++) far[j] = cin[u[j] >= hub_n ? u[j] : 0];
#pragma unroll
  for (int j = 0; j < kN; j++) near[j] = hub[u[j] < hub_n ? u[j] : 0];
#pragma unroll
  for (int j = 0; j < kN; j++) x[j] = k + j * stride >= e ? T(0) : u[j] >= hub_n ? far[j] : near[j];
}

// ---- FP32_SERIAL ----------------------------------------------------------
//
// The reference's arithmetic: each row's contributions added one by one in
// FP32, in in-neighbour order (src/pr.cc:57-59).  The order of the additions
// is fixed, not who does them; rows are taken by length:
//   bundles      kLightBundle rows (below heavy_threshold) or kHeavyBundle
//                rows per wavefront, gathered together and coalesced, one
//                lane adding each row
//   long rows    from kSerialWaveRow on by a wavefront, from kSerialBlockRow
//                on by a workgroup, by exact composition (serial_fold)
// What bounds it: the gathers beyond the LDS hub, some 200 G/s (a cache line
// into L1 for each), and per CU about 1/256 of that, so items are dealt to
// the CUs by their edges (serial_plan).  Kronecker-21, per iteration that runs:
// 262 us (242 G edges/s, those that the hub serves included); 6.12 ms with a
// wavefront per heavy row adding shuffled values one by one (the longest row,
// some 10^5 edges, took that long).  A whole rank of 7 iterations, when the
// items came: 2.42 ms, strided over small workgroups without the hub 2.67,
// strided with it 2.9.
//
// Long rows by composition.  While the running sum S stays inside one binade
// [2^E, 2^(E+1)), S is an integer multiple of u = 2^(E-23), and adding x >= 0
// adds the integer rn(x / u), except that an exact half goes to the even
// neighbour, which depends only on the parity of S / u.  So every run of
// additions inside a binade is a pair (what it adds to an even S, to an odd
// S), and pairs compose associatively: lanes build their own kSerialPer
// elements' pairs and a scan over the wavefront composes them, in order, with
// exact integers.  The element where S leaves the binade is found from the
// scan; the lane that holds it adds its elements one by one, and the scan
// goes on behind that lane with the new binade.  S only grows, so a row of d
// elements crosses at most about log2(d) + 30 binades.  Negative or non-finite
// contributions, and sums below 2^-103, are added one lane after another.

constexpr int kSerialThreads = 1024;
constexpr int kSerialWaves = kSerialThreads / 64;
constexpr int kSerialHub = 28672;         // contributions in LDS (112 KB, whole 16-byte loads per thread)
constexpr int kSerialPer = 8;             // edges per lane and step
constexpr int kHeavyCols = 64 * kSerialPer / kHeavyBundle;  // edges of each row per step of a bundle
constexpr int kLightCols = 64 * kSerialPer / kLightBundle;
constexpr int kHeavyPitch = kHeavyCols + 4;  // LDS floats from row to row: no two rows of a read on one bank
constexpr int kLightPitch = kLightCols + 2;
constexpr int kStageFloats = kHeavyBundle * kHeavyPitch > kLightBundle * kLightPitch ? kHeavyBundle * kHeavyPitch
                                                                                     : kLightBundle * kLightPitch;
constexpr unsigned kBinadeEnd = 1u << 24;

__device__ __forceinline__ float lane_value(float x, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}

// Whether composition works from S: positive, normal, both its unit and the
// reciprocal of the unit normal.
__device__ __forceinline__ bool composable(float S) {
  const unsigned eb = __float_as_uint(S) >> 23;  // a set sign bit makes it >= 256
  return eb >= 24u && eb <= 254u;
}
__device__ __forceinline__ unsigned units_of(float S) { return (__float_as_uint(S) & 0x7FFFFFu) | 0x800000u; }
// The float of `units` (below kBinadeEnd) in S's binade.
__device__ __forceinline__ float from_units(float S, unsigned units) {
  return __uint_as_float((__float_as_uint(S) & 0xFF800000u) | (units & 0x7FFFFFu));
}

__device__ __forceinline__ bool all_plain(const float (&x)[kSerialPer]) {
  bool ok = true;
#pragma unroll
  for (int j = 0; j < kSerialPer; j++) ok = ok && x[j] >= 0.0f && x[j] < __builtin_inff();
  return __ballot(!ok) == 0ull;
}

// The lane's pair under S's unit: what its elements add to an even and to an
// odd multiple, each saturated at kBinadeEnd (past any binade's end).
__device__ __forceinline__ void lane_pair(float S, const float (&x)[kSerialPer], unsigned& a0, unsigned& a1) {
  const float scale = __uint_as_float((277u - (__float_as_uint(S) >> 23)) << 23);  // 1 / u
  a0 = a1 = 0;
#pragma unroll
  for (int j = 0; j < kSerialPer; j++) {
    const float t = fminf(x[j] * scale, 16777216.0f);  // exact below the clamp (or far below one half)
    const float r = rintf(t);                          // half to even
    const float d = t - r;
    const unsigned c0 = static_cast<unsigned>(r);
    const unsigned c1 = fabsf(d) == 0.5f ? static_cast<unsigned>(t + d) : c0;  // the other neighbour of a half
    a0 += (a0 & 1u) ? c1 : c0;
    a1 += (a1 & 1u) ? c0 : c1;
  }
  a0 = min(a0, kBinadeEnd);
  a1 = min(a1, kBinadeEnd);
}

// Inclusive scan over the lanes of what they add to S (its parity is
// `odd`).  Without halves (both entries equal in every lane) a plain sum.
__device__ __forceinline__ unsigned pair_scan(unsigned a0, unsigned a1, unsigned odd) {
  if (__ballot(a0 != a1) == 0ull) return wave_scan_u32(a0);
  const int lane = lane_id();
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const unsigned p0 = __shfl_up(a0, d, 64), p1 = __shfl_up(a1, d, 64);
    if (lane >= d) {
      const unsigned n0 = p0 + ((p0 & 1u) ? a1 : a0);
      const unsigned n1 = p1 + ((p1 & 1u) ? a0 : a1);
      a0 = n0;
      a1 = n1;
    }
  }
  return odd ? a1 : a0;
}

// S after adding the wavefront's elements in lane order (lane i holds the
// elements [i * kSerialPer, (i + 1) * kSerialPer)); S is wave-uniform.
__device__ __forceinline__ float serial_fold(float S, const float (&x)[kSerialPer], int lane) {
  const bool plain = all_plain(x);
  for (int from = 0; from < 64;) {
    int at = from;  // the lane whose elements are added one by one
    if (plain && composable(S)) {
      unsigned a0, a1;
      lane_pair(S, x, a0, a1);
      if (lane < from) a0 = a1 = 0;
      const unsigned si = units_of(S);
      const unsigned incl = pair_scan(a0, a1, si & 1u);
      const unsigned long long over = __ballot(si + incl >= kBinadeEnd);
      if (over == 0ull) return from_units(S, si + __builtin_amdgcn_readlane(incl, 63));
      at = __builtin_ctzll(over);
      if (at > from) S = from_units(S, si + __builtin_amdgcn_readlane(incl, at - 1));
    }
    float r = S;
#pragma unroll
    for (int j = 0; j < kSerialPer; j++) r += x[j];
    S = lane_value(r, at);
    from = at + 1;
  }
  return S;
}

// The contributions of the first n vertices, in LDS, and a zero behind the
// room for them.
struct SerialHub {
  const float* lds;
  int n;
};

// The contributions of kSerialPer edges on their way.  A wavefront's loads
// are unconditional (lanes without work read a spare place), so that every
// path issues the same number: a step's IDs are waited for with the previous
// step's gathers in flight, and its gathers with the next step's.
struct SerialStep {
  int32_t v[kSerialPer];  // sources, -1: no edge
  float g[kSerialPer];    // what lies beyond the hub
  __device__ __forceinline__ void load(const SerialHub& hub, const float* __restrict__ cin) {
#pragma unroll
    for (int j = 0; j < kSerialPer; j++) g[j] = cin[v[j] >= hub.n ? v[j] : 0];
  }
  __device__ __forceinline__ void take(const SerialHub& hub, float (&x)[kSerialPer]) const {
    float l[kSerialPer];
#pragma unroll
    for (int j = 0; j < kSerialPer; j++)
      l[j] = hub.lds[static_cast<unsigned>(v[j]) < static_cast<unsigned>(hub.n) ? v[j] : kSerialHub];
    // No edge adds +0, which changes no sum here (they start at +0).
#pragma unroll
    for (int j = 0; j < kSerialPer; j++) x[j] = v[j] >= hub.n ? g[j] : l[j];
  }
};

// Source IDs of in-edges [k, k + kSerialPer) of a row that ends at e and has
// at least kSerialPer: past the end the last kSerialPer, of which keep_ids
// drops the ones below k.
__device__ __forceinline__ void load_ids(const int32_t* __restrict__ nbr, int64_t k, int64_t e,
                                         int32_t (&v)[kSerialPer]) {
  __builtin_memcpy(v, nbr + min(k, e - kSerialPer), sizeof(v));  // rows start at any 4-byte address
}
__device__ __forceinline__ void keep_ids(int64_t k, int64_t e, const int32_t (&raw)[kSerialPer], SerialStep& st) {
  const int drop = static_cast<int>(max<int64_t>(0, min<int64_t>(kSerialPer, k - (e - kSerialPer))));
#pragma unroll
  for (int j = 0; j < kSerialPer; j++) st.v[j] = j >= drop ? raw[j] : -1;
}

// The steps of one row, kLanes lanes wide, handed to f(x) in order.
template <int kLanes, typename F>
__device__ __forceinline__ void row_steps(const int32_t* __restrict__ nbr, const SerialHub& hub,
                                          const float* __restrict__ cin, int64_t s, int64_t e, int lane, F&& f) {
  constexpr int64_t kStep = int64_t(kLanes) * kSerialPer;
  int64_t k = s + int64_t(lane) * kSerialPer;
  int32_t raw[kSerialPer];
  SerialStep cur, next;
  load_ids(nbr, k, e, raw);
  keep_ids(k, e, raw, cur);
  load_ids(nbr, k + kStep, e, raw);
  cur.load(hub, cin);
  for (int64_t at = s; at < e; at += kStep) {
    k += kStep;
    keep_ids(k, e, raw, next);
    load_ids(nbr, k + kStep, e, raw);
    next.load(hub, cin);
    float x[kSerialPer];
    cur.take(hub, x);
    f(x);
    cur = next;
  }
}

struct SerialLds {
  float hub[kSerialHub + 4];
  float stage[kSerialWaves][kStageFloats];
  unsigned p0[2][kSerialWaves], p1[2][kSerialWaves];
  float sum[2];
  double red[kSerialWaves + 1];
};
static_assert(sizeof(SerialLds) <= 160 * 1024, "one workgroup per CU");

// A very long row by the workgroup.  Each round every wavefront not yet
// folded in offers the pair of its elements under the sum's binade; they are
// taken in wave order until one would leave the binade, which that wavefront
// then folds itself.
__device__ __forceinline__ float serial_block_row(const PrArgs& a, const SerialHub& hub,
                                                  const float* __restrict__ cin, int64_t s, int64_t e, SerialLds& L) {
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float S = 0.0f;
  int buf = 0;  // the exchange words alternate, so one barrier separates their uses
  row_steps<kSerialThreads>(a.in_nbr, hub, cin, s, e, threadIdx.x, [&](const float (&x)[kSerialPer]) {
    const bool plain = all_plain(x);
    for (int from = 0; from < kSerialWaves;) {
      const bool can = composable(S);  // the same in every wavefront
      if (can && wave >= from) {
        unsigned a0 = kBinadeEnd, a1 = kBinadeEnd;
        if (plain) {
          unsigned l0, l1;
          lane_pair(S, x, l0, l1);
          if (__ballot(l0 != l1) == 0ull) {
            a0 = a1 = __builtin_amdgcn_readlane(wave_scan_u32(l0), 63);
          } else {
            a0 = __builtin_amdgcn_readlane(pair_scan(l0, l1, 0u), 63);
            a1 = __builtin_amdgcn_readlane(pair_scan(l0, l1, 1u), 63);
          }
        }
        if (lane == 0) {
          L.p0[buf][wave] = min(a0, kBinadeEnd);
          L.p1[buf][wave] = min(a1, kBinadeEnd);
        }
      }
      __syncthreads();
      if (can) {
        unsigned si = units_of(S);
        for (; from < kSerialWaves; from++) {
          const unsigned add = (si & 1u) ? L.p1[buf][from] : L.p0[buf][from];
          if (si + add >= kBinadeEnd) break;
          si += add;
        }
        S = from_units(S, si);
      }
      if (from < kSerialWaves) {
        if (wave == from) {
          const float r = serial_fold(S, x, lane);
          if (lane == 0) L.sum[buf] = r;
        }
        __syncthreads();
        S = L.sum[buf];
        from++;
      }
      buf ^= 1;
    }
  });
  __syncthreads();  // the exchange words are free for the next row
  return S;
}

// kRows rows by one wavefront, lane i adding the row [s, s + len) it holds
// (len 0: none): the wavefront gathers kCols edges of every row at a time
// and stages them in LDS.  Returns the lane's sum.
template <int kRows, int kCols, int kPitch>
__device__ __forceinline__ float serial_bundle(const int32_t* __restrict__ nbr, const SerialHub& hub,
                                               const float* __restrict__ cin, int64_t s, int len, int lane,
                                               float* stage) {
  static_assert(kRows * kCols == 64 * kSerialPer, "a step's edges");
  constexpr int kPass = 64 / kCols;  // rows per load
  const int col = lane % kCols;
  int64_t base[kSerialPer];
  int left[kSerialPer];
#pragma unroll
  for (int j = 0; j < kSerialPer; j++) {
    const int r = j * kPass + lane / kCols;
    base[j] = __shfl(s, r, 64) + col;
    left[j] = __shfl(len, r, 64) - col;
  }
  int longest = len;
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) longest = max(longest, __shfl_xor(longest, d, 64));
  longest = __builtin_amdgcn_readfirstlane(longest);
  int32_t raw[kSerialPer];
  SerialStep cur, next;
  auto load = [&](int c) {
#pragma unroll
    for (int j = 0; j < kSerialPer; j++) raw[j] = nbr[c < left[j] ? base[j] + c : 0];
  };
  auto keep = [&](int c, SerialStep& st) {
#pragma unroll
    for (int j = 0; j < kSerialPer; j++) st.v[j] = c < left[j] ? raw[j] : -1;
  };
  if (longest == 0) return 0.0f;
  load(0);
  keep(0, cur);
  load(kCols);
  cur.load(hub, cin);
  float sum = 0.0f;
  using Quad = float __attribute__((ext_vector_type(kPitch % 4 == 0 ? 4 : 2)));
  constexpr int kQuad = sizeof(Quad) / 4;
  const Quad* mine = reinterpret_cast<const Quad*>(stage + (lane % kRows) * kPitch);
  float* put = stage + (lane / kCols) * kPitch + col;
  for (int c = 0; c < longest; c += kCols) {
    keep(c + kCols, next);
    load(c + 2 * kCols);
    next.load(hub, cin);
    float x[kSerialPer];
    cur.take(hub, x);
    // LDS operations of one wavefront complete in order: only the compiler's
    // order needs holding between the writes and the other lanes' reads.
#pragma unroll
    for (int j = 0; j < kSerialPer; j++) put[j * kPass * kPitch] = x[j];
    __asm__ volatile("" ::: "memory");
#pragma unroll
    for (int q = 0; q < kCols / kQuad; q++) {
      const Quad z = mine[q];
#pragma unroll
      for (int i = 0; i < kQuad; i++) sum += z[i];
    }
    __asm__ volatile("" ::: "memory");
    cur = next;
  }
  return sum;
}

// One iteration, one workgroup per CU: it fills its hub, takes its very long
// rows, its wavefronts take the rest of its items in turn, and the rows
// without in-edges go to all threads.
__global__ __launch_bounds__(kSerialThreads) void k_serial(PrArgs a, PrPrev prev, const float* __restrict__ cin,
                                                           float* __restrict__ cout, float* __restrict__ score) {
  __shared__ SerialLds L;
  if (!pr_begin<kSerialThreads>(prev, L.red)) return;
  const SerialHub hub{L.hub, a.serial_hub};
  if (hub.n > 0) lds_fill<float, kSerialHub * 4, kSerialThreads>(L.hub, cin, hub.n);
  if (threadIdx.x == 0) L.hub[kSerialHub] = 0.0f;
  __syncthreads();
  double err = 0;
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int i = a.sstart[blockIdx.x];
  const int end = a.sstart[blockIdx.x + 1];
  for (; i < end && a.sitems[i].kind == kSerialBlock; i++) {
    const int64_t u = a.sitems[i].first;
    const float sum = serial_block_row(a, hub, cin, a.in_off[u], a.in_off[u + 1], L);
    if (threadIdx.x == 0) err += finish_f32(a, u, sum, score, cout);
  }
  for (i += wave; i < end; i += kSerialWaves) {
    const SerialItem it = a.sitems[i];
    if (it.kind == kSerialWave) {
      const int64_t s = a.in_off[it.first], e = a.in_off[it.first + 1];
      float sum = 0.0f;
      row_steps<64>(a.in_nbr, hub, cin, s, e, lane,
                    [&](const float (&x)[kSerialPer]) { sum = serial_fold(sum, x, lane); });
      if (lane == 0) err += finish_f32(a, it.first, sum, score, cout);
      continue;
    }
    // Rows of the heavy list, or neighbouring rows of which the heavy ones
    // are someone else's.
    const bool heavy = it.kind == kSerialHeavy;
    const int64_t at = int64_t(it.first) + lane;
    int64_t row = -1;
    if (heavy) {
      if (lane < kHeavyBundle && at < a.n_heavy) row = a.heavy[at];
    } else if (at < a.zero_begin) {
      row = at;
    }
    int64_t s = 0;
    int len = 0;
    if (row >= 0) {
      s = a.in_off[row];
      const int64_t d = a.in_off[row + 1] - s;
      if (!heavy && d >= a.heavy_threshold)
        row = -1;
      else
        len = static_cast<int>(d);
    }
    const float sum =
        heavy ? serial_bundle<kHeavyBundle, kHeavyCols, kHeavyPitch>(a.in_nbr, hub, cin, s, len, lane, L.stage[wave])
              : serial_bundle<kLightBundle, kLightCols, kLightPitch>(a.in_nbr, hub, cin, s, len, lane, L.stage[wave]);
    if (row >= 0) err += finish_f32(a, row, sum, score, cout);
  }
  for (int64_t u = a.zero_begin + int64_t(blockIdx.x) * kSerialThreads + threadIdx.x; u < a.nloc;
       u += int64_t(gridDim.x) * kSerialThreads)
    err += finish_f32(a, u, 0.0f, score, cout);
  const double t = block_err_sum<kSerialThreads>(err, L.red);
  if (threadIdx.x == 0) a.err_part[blockIdx.x] = t;
}

// ---- FP32_KAHAN -------------------------------------------------------------

// Compensated FP32 / plain FP64 sums, one fused launch per iteration.
//
// Persistent blocks of kFusedThreads (one per CU).  Each block first copies
// the contributions of vertices [0, hub_n) -- 128 KB -- into LDS; in the
// degree-ordered layout these are the highest-degree vertices and receive
// about half of all gathers on Kronecker graphs, which LDS serves several
// times faster than L2.  Wavefronts then take the heavy items (rows with
// in-degree >= heavy_threshold, or 2048-edge segments of split rows), one
// item per wave with lanes striding its edge range and kUnroll gathers in
// flight, afterwards the light rows in kGroup-lane groups, and last the rows
// without in-edges, one per thread.  A split row's segments store
// (sum, error) pairs for the combine kernel.
//
// What bounds it: the gathers beyond the hub where they miss L2 (3.7 M or
// 1.9 M uniform vertices: 64 to 70 G/s of lines), else the latency of a row's
// chain of loads, so no row takes its edges one step at a time: what is left
// of an item and a light row's edges are masked steps, and light rows are
// pipelined.  FP64, 20 iterations, whole call: Kronecker 1.7 M 4.00 -> 3.59 ms
// (the light rows 3.79; an item's rest in steps of 2, 4, 8 edges a lane 3.68,
// 3.59, 3.63), 1.9 M uniform 16.45 -> 16.09, 60 K the same.  Items pipelined
// like the light rows: 3.65 and 60 K 18% slower.
template <typename T>
struct FusedAcc;

template <>
struct FusedAcc<float> {
  Comp c{0.0f, 0.0f};
  __device__ __forceinline__ void add(float x) { c.add(x); }
  // Fixed butterfly merge; operands ordered by lane so both partners of a
  // pair compute the same value.
  template <int kWidth>
  __device__ __forceinline__ void reduce(int sub) {
#pragma unroll
    for (int d = kWidth / 2; d >= 1; d >>= 1) {
      const float s2 = __shfl_xor(c.s, d, kWidth);
      const float c2 = __shfl_xor(c.c, d, kWidth);
      if (sub & d) {
        Comp o{s2, c2};
        o.merge(c.s, c.c);
        c = o;
      } else {
        c.merge(s2, c2);
      }
    }
  }
  __device__ __forceinline__ float value() const { return c.value(); }
  __device__ __forceinline__ double2 partial() const { return make_double2(c.s, c.c); }
  __device__ __forceinline__ void merge(float2 p) { c.merge(p.x, p.y); }
};

template <>
struct FusedAcc<double> {
  double s = 0.0;
  __device__ __forceinline__ void add(double x) { s += x; }
  template <int kWidth>
  __device__ __forceinline__ void reduce(int) {
#pragma unroll
    for (int d = kWidth / 2; d >= 1; d >>= 1) s += __shfl_xor(s, d, kWidth);
  }
  __device__ __forceinline__ double value() const { return s; }
  __device__ __forceinline__ double2 partial() const { return make_double2(s, 0.0); }
};

__device__ __forceinline__ double finish_t(const PrArgs& a, int64_t lu, float in, float* score, float* cout) {
  return finish_f32(a, lu, in, score, cout);
}
__device__ __forceinline__ double finish_t(const PrArgs& a, int64_t lu, double in, double* score, double* cout) {
  return finish_f64(a, lu, in, score, cout);
}

template <typename T>
__device__ __forceinline__ T base_t(const PrArgs& a) {
  if constexpr (sizeof(T) == 8) return a.prm->base_d; else return a.prm->base_f;
}
template <typename T>
__device__ __forceinline__ T damp_t(const PrArgs& a) {
  if constexpr (sizeof(T) == 8) return a.prm->damp_d; else return a.prm->damp_f;
}
__device__ __forceinline__ float abs_t(float x) { return fabsf(x); }
__device__ __forceinline__ double abs_t(double x) { return fabs(x); }

template <typename T>
__global__ __launch_bounds__(kFusedThreads) void k_fused(PrArgs a, PrPrev prev, const T* __restrict__ cin,
                                                         T* __restrict__ cout, T* __restrict__ score) {
  __shared__ T hub[kHubBytes / sizeof(T)];
  __shared__ double red[kFusedThreads / 64 + 1];
  if (!pr_begin<kFusedThreads>(prev, red)) return;
  const int hub_n = static_cast<int>(min<int64_t>(kHubBytes / sizeof(T), a.n_gather));
  lds_fill<T, kHubBytes>(hub, cin, hub_n);
  __syncthreads();

  double err = 0;
  const int lane = lane_id();
  const T base = base_t<T>(a), damp = damp_t<T>(a);
  auto finish = [&](int64_t u, T sum, T old, int64_t deg) {
    const T nw = base + damp * sum;
    score[u] = nw;
    cout[u] = nw / static_cast<T>(deg);
    err += static_cast<double>(abs_t(nw - old));
  };
  // Heavy items, one per wavefront, kUnroll edges a lane and step.
  const int64_t wave = (int64_t(blockIdx.x) * kFusedThreads + threadIdx.x) >> 6;
  const int64_t nwaves = (int64_t(gridDim.x) * kFusedThreads) >> 6;
  for (int64_t h = wave; h < a.n_items; h += nwaves) {
    const PrItem it = a.items[h];
    FusedAcc<T> acc;
    T x[kUnroll];
    int32_t u[kUnroll];
    int64_t k = it.b + lane;
    for (; k + 64 * (kUnroll - 1) < it.e; k += 64 * kUnroll) {
#pragma unroll
      for (int j = 0; j < kUnroll; j++) u[j] = a.in_nbr[k + 64 * j];
      hub_gathers(hub, hub_n, cin, u, k, 64, it.e, x);
#pragma unroll
      for (int j = 0; j < kUnroll; j++) acc.add(x[j]);
    }
    for (; k < it.e; k += 64 * kTailUnroll) {
      int32_t v[kTailUnroll];
      T y[kTailUnroll];
#pragma unroll
      for (int j = 0; j < kTailUnroll; j++) v[j] = k + 64 * j < it.e ? a.in_nbr[k + 64 * j] : 0;
      hub_gathers(hub, hub_n, cin, v, k, 64, it.e, y);
#pragma unroll
      for (int j = 0; j < kTailUnroll; j++) acc.add(y[j]);
    }
    acc.template reduce<64>(lane);
    if (lane == 0) {
      if (it.slot < 0)
        finish(it.v, acc.value(), score[it.v], out_deg(a, it.v));
      else
        a.partial[it.slot] = acc.partial();
    }
  }
  // Light rows, one per kGroup-lane group; every lane of a wavefront runs the
  // same number of rounds so the group shuffles stay convergent.  A row is a
  // chain of bounds, neighbours, contributions and its old score; while one
  // row's contributions arrive, the next row's neighbours (kLightUnroll a
  // lane) and score and the bounds of the row after it are on their way.
  // They are waited for before the row's stores: loads and stores complete in
  // issue order.  Two buffers alternate, so that no copy waits.
  const int sub = threadIdx.x & (kGroup - 1);
  const int64_t grp = (int64_t(blockIdx.x) * kFusedThreads + threadIdx.x) / kGroup;
  const int64_t ngrp = (int64_t(gridDim.x) * kFusedThreads) / kGroup;
  const int64_t rounds = (a.light_end - a.light_begin + ngrp - 1) / ngrp;
  struct Bounds {
    int64_t s, e;
  };
  struct Row {
    int64_t o0, o1;
    T old;
    int32_t v[kLightUnroll];
    bool mine;
  };
  auto load_bounds = [&](int64_t r) {
    const int64_t u = a.light_begin + grp + r * ngrp;
    Bounds b{0, a.heavy_threshold};
    if (u < a.light_end) {
      b.s = a.in_off[u];
      b.e = a.in_off[u + 1];
    }
    return b;
  };
  auto load_light = [&](int64_t k, int64_t e, int32_t (&v)[kLightUnroll]) {
#pragma unroll
    for (int j = 0; j < kLightUnroll; j++) v[j] = k + j * kGroup < e ? a.in_nbr[k + j * kGroup] : 0;
  };
  auto load_row = [&](int64_t r, const Bounds& b, Row& n) {
    const int64_t u = a.light_begin + grp + r * ngrp;
    n.mine = b.e - b.s < a.heavy_threshold;
    load_light(b.s + sub, n.mine ? b.e : b.s, n.v);
    n.old = T(0);
    n.o0 = n.o1 = 0;
    if (n.mine && sub == 0) {
      n.old = score[u];
      n.o0 = a.out_off[u];
      n.o1 = a.out_off[u + 1];
    }
  };
  // Row r, its bounds in hb (which then take row r + 2's), the next row's in hn.
  auto light = [&](int64_t r, Bounds& hb, const Row& row, const Bounds& hn, Row& next) {
    const Bounds b{hb.s, row.mine ? hb.e : hb.s};
    load_row(r + 1, hn, next);
    hb = load_bounds(r + 2);
    FusedAcc<T> acc;
    T x[kLightUnroll];
    hub_gathers(hub, hub_n, cin, row.v, b.s + sub, kGroup, b.e, x);
#pragma unroll
    for (int j = 0; j < kLightUnroll; j++) acc.add(x[j]);
    for (int64_t k = b.s + kLightUnroll * kGroup + sub; k - sub < b.e; k += kLightUnroll * kGroup) {
      int32_t v[kLightUnroll];
      load_light(k, b.e, v);
      hub_gathers(hub, hub_n, cin, v, k, kGroup, b.e, x);
#pragma unroll
      for (int j = 0; j < kLightUnroll; j++) acc.add(x[j]);
    }
    acc.template reduce<kGroup>(sub);
#pragma unroll
    for (int j = 0; j < kLightUnroll; j++) __asm__ volatile("" ::"v"(next.v[j]) : "memory");
    __asm__ volatile("" ::"v"(next.old), "v"(next.o0), "v"(next.o1), "v"(hb.s), "v"(hb.e) : "memory");
    if (row.mine && sub == 0) finish(a.light_begin + grp + r * ngrp, acc.value(), row.old, row.o1 - row.o0);
  };
  Bounds ha = load_bounds(0), hb = load_bounds(1);
  Row ra, rb;
  load_row(0, ha, ra);
  for (int64_t r = 0; r < rounds; r += 2) {
    light(r, ha, ra, hb, rb);
    if (r + 1 >= rounds) break;
    light(r + 1, hb, rb, ha, ra);
  }
  // Rows without in-edges: the empty sum.
  for (int64_t u = a.zero_begin + int64_t(blockIdx.x) * kFusedThreads + threadIdx.x; u < a.nloc;
       u += int64_t(gridDim.x) * kFusedThreads)
    err += finish_t(a, u, T(0), score, cout);
  const double t = block_err_sum<kFusedThreads>(err, red);
  if (threadIdx.x == 0) a.err_part[blockIdx.x] = t;
}

// ---- FP32_KAHAN, window-tiled (degree-ordered whole graphs) ----------------

template <int kCtrl, int kRowMask>
__device__ __forceinline__ double dpp_move(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(b), kCtrl, kRowMask, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), kCtrl, kRowMask, 0xf, true);
  return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned int>(lo));
}

// Inclusive scan of v over lanes [seg, lane] (seg = the lane's segment
// head), from DPP lane moves: row_shr 1/2/4/8 inside 16-lane rows, then
// row_bcast 15 and 31 across rows.
__device__ __forceinline__ double seg_scan(double v, int lane, int seg) {
  double t;
  t = dpp_move<0x111, 0xf>(v);  // row_shr:1
  if ((lane & 15) >= 1 && lane - 1 >= seg) v += t;
  t = dpp_move<0x112, 0xf>(v);  // row_shr:2
  if ((lane & 15) >= 2 && lane - 2 >= seg) v += t;
  t = dpp_move<0x114, 0xf>(v);  // row_shr:4
  if ((lane & 15) >= 4 && lane - 4 >= seg) v += t;
  t = dpp_move<0x118, 0xf>(v);  // row_shr:8
  if ((lane & 15) >= 8 && lane - 8 >= seg) v += t;
  t = dpp_move<0x142, 0xa>(v);  // row_bcast:15 -> rows 1 and 3 get lanes 15 / 47
  if (((lane >> 4) & 1) && (lane & ~15) - 1 >= seg) v += t;
  t = dpp_move<0x143, 0xc>(v);  // row_bcast:31 -> rows 2 and 3 get lane 31
  if (lane >= 32 && 31 >= seg) v += t;
  return v;
}

struct TileArgs {
  const int32_t* cwin;     // window of each chunk
  const int64_t* wstart;   // first chunk of each window (+ end)
  const int32_t* cbase;    // first partial of each chunk (+ end)
  const uint32_t* meta;    // per lane: end mask | filled slots << 16
  const uint16_t* src;
  int64_t n_chunks;
  float* part;             // per piece: its FP64 sum rounded to FP32
  const int32_t* brow;     // row blocks: first row (+ end)
  const int64_t* bseg;     //             first segment (+ end)
  const int32_t* bsize;    //             partials (the region's size)
  const int32_t* seg_start;  // segments: first partial
  const int32_t* seg_off;    //           offset in the block's region
  const int32_t* istart;   // per row: first list entry (+ end)
  const uint16_t* idx;     // per row: partial offsets in its block's region, window order
  int64_t n_blocks;
};

constexpr int kTileThreads = 1024;

// What one lane reads of a chunk from HBM: its end mask / slot count, its
// kLaneEdges 16-bit source offsets and the chunk's partial range.
struct ChunkLoad {
  uint32_t mt;
  uint4 q0, q1;
  int32_t c0, c1;
};

__device__ __forceinline__ ChunkLoad load_chunk(const TileArgs& t, int64_t c, int lane) {
  ChunkLoad l;
  l.mt = t.meta[c * 64 + lane];
  const uint4* s4 = reinterpret_cast<const uint4*>(t.src + c * kChunkEdges + lane * kLaneEdges);
  l.q0 = s4[0];
  l.q1 = s4[1];
  l.c0 = t.cbase[c];
  l.c1 = t.cbase[c + 1];
  return l;
}

// One chunk of the tile pass, run by one wavefront.  Lane i holds slots
// [i * kLaneEdges, (i + 1) * kLaneEdges) of the chunk; a piece may span
// lanes but never chunks.  First pass: each lane sums its edges after its
// last piece end (all of them if none ends in it).  A segmented scan of
// these tails over the lanes (restarted at lanes where a piece ends) gives
// each lane the carry of the piece still open at its start.  Second pass:
// the lane sums its edges again from the carry, restarting at every piece
// end, where a piece is complete.  Values accumulate in FP64 (a piece holds
// at most kChunkEdges FP32 values, relative error <= kChunkEdges * 2^-53)
// and a piece enters its row's compensated FP32 sum rounded to FP32 (half
// a unit in its last place).  Every term of a row's sum is non-negative, so
// these roundings add at most one unit in the last place of the row's sum.
//
// Slots past a lane's filled count are not masked: every chunk closes its
// last piece at its last filled slot, so those slots (which read offset 0)
// lie after the chunk's last piece end and reach no piece.
//
// The chunk's pieces (at most kChunkPieces), numbered in lane order, are
// staged, rounded to FP32, in the wavefront's LDS area and written to the
// chunk's contiguous partial range by kChunkPieces / 64
// store instructions of consecutive lanes.  With that fixed count, a chunk whose loads were issued before
// these stores is waited for without waiting for the stores (vector memory
// operations complete in issue order).
__device__ __forceinline__ void tile_chunk(const TileArgs& t, const float* win, ChunkLoad l, int lane,
                                           float* stage) {
  // Every use of the chunk's loaded registers stays after the previous
  // chunk's stores (the asm is ordered with memory operations), so the
  // compiler cannot move one early into a wait that covers those stores.
  __asm__ volatile(""
                   : "+v"(l.mt), "+v"(l.q0.x), "+v"(l.q0.y), "+v"(l.q0.z), "+v"(l.q0.w), "+v"(l.q1.x), "+v"(l.q1.y),
                     "+v"(l.q1.z), "+v"(l.q1.w), "+v"(l.c0), "+v"(l.c1)
                   :
                   : "memory");
  const uint32_t sw[8] = {l.q0.x, l.q0.y, l.q0.z, l.q0.w, l.q1.x, l.q1.y, l.q1.z, l.q1.w};
  const uint32_t ends = l.mt & 0xFFFFu;
  double x[kLaneEdges];
#pragma unroll
  for (int j = 0; j < kLaneEdges; j++) x[j] = static_cast<double>(win[(sw[j >> 1] >> (16 * (j & 1))) & 0xFFFFu]);
  // The lane's last piece end (-1 if none): its tail is the sum after it.
  const int last = ends ? 31 - __builtin_clz(ends) : -1;
  double acc = 0.0;
#pragma unroll
  for (int j = 0; j < kLaneEdges; j++) acc += j > last ? x[j] : 0.0;
  const unsigned long long has_end = __ballot(ends != 0u);
  const unsigned long long upto = lane == 63 ? ~0ull : ((2ull << lane) - 1);
  const unsigned long long h = has_end & upto;
  const int seg = h ? 63 - __clzll(static_cast<long long>(h)) : 0;
  const double carry_out = seg_scan(acc, lane, seg);
  double a = __shfl_up(carry_out, 1, 64);
  if (lane == 0) a = 0.0;
  const uint32_t k_i = __builtin_popcount(ends);
  // Second pass: the lanes where a piece ends at slot j write it to its
  // staging entry and restart.
  float* qq = stage + (wave_scan_u32(k_i) - k_i);  // the lane's first piece
#pragma unroll
  for (int j = 0; j < kLaneEdges; j++) {
    a += x[j];
    if ((ends >> j) & 1u) {
      *qq++ = static_cast<float>(a);
      a = 0.0;
    }
  }
  // The staged pieces are read back by other lanes of this wavefront; LDS
  // operations of one wavefront complete in issue order, so only the
  // compiler's order needs holding here.
  __asm__ volatile("" ::: "memory");
  // Always kChunkPieces / 64 stores, with no branch around them: lanes past
  // the chunk's last piece write that piece again.  The chunk's first
  // partial and piece count are wave-uniform: the stores take a scalar base.
  const int32_t c0 = __builtin_amdgcn_readfirstlane(l.c0);
  const int np = __builtin_amdgcn_readfirstlane(l.c1) - c0;
  float* const dst = t.part + c0;
  float v[kChunkPieces / 64];
#pragma unroll
  for (int r = 0; r < kChunkPieces / 64; r++) v[r] = stage[min(lane + 64 * r, np - 1)];
#pragma unroll
  for (int r = 0; r < kChunkPieces / 64; r++) dst[min(lane + 64 * r, np - 1)] = v[r];
  __asm__ volatile("" ::: "memory");  // the next chunk's staging follows these reads
}

// Waits for a chunk's loads (used where no vector memory operation follows
// them, so that the wait there does not cover later stores).
__device__ __forceinline__ void chunk_ready(const ChunkLoad& l) {
  __asm__ volatile("" ::"v"(l.mt), "v"(l.q0.x), "v"(l.q0.y), "v"(l.q0.z), "v"(l.q0.w), "v"(l.q1.x), "v"(l.q1.y),
                   "v"(l.q1.z), "v"(l.q1.w), "v"(l.c0), "v"(l.c1));
}

// Tile pass: persistent workgroups (one per CU), each owning a contiguous
// range of chunks (window-major); the workgroup copies one window of
// contributions into LDS at a time and its wavefronts take the window's
// chunks in turn, each loading its next chunk before it sums the current.
template <int kWin>
__global__ __launch_bounds__(kTileThreads) void k_tile(TileArgs t, PrPrev prev, const float* __restrict__ cin,
                                                      int64_t n_gather) {
  __shared__ float win[kWin];
  __shared__ __align__(8) float stage_all[kTileThreads / 64][kChunkPieces];
  if (!pr_begin<kTileThreads>(prev, reinterpret_cast<double*>(stage_all))) return;
  const int64_t per = (t.n_chunks + gridDim.x - 1) / gridDim.x;
  const int64_t c0 = min(t.n_chunks, int64_t(blockIdx.x) * per), c1 = min(t.n_chunks, c0 + per);
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform: scalar chunk indices
  float* stage = stage_all[wave];
  constexpr int kWaves = kTileThreads / 64;
  for (int64_t c = c0; c < c1;) {
    const int32_t w = t.cwin[c];
    const int64_t wend = min(c1, t.wstart[w + 1]);
    const int64_t base = int64_t(w) * kWin;
    const int cnt = static_cast<int>(min<int64_t>(kWin, n_gather - base));
    __syncthreads();  // the previous window's readers are done
    if (cnt == kWin) {
      const float4* s = reinterpret_cast<const float4*>(cin + base);
      float4* d = reinterpret_cast<float4*>(win);
      constexpr int kPer = kWin / 4 / kTileThreads;
      float4 v[kPer];
#pragma unroll
      for (int i = 0; i < kPer; i++) v[i] = s[threadIdx.x + i * kTileThreads];
#pragma unroll
      for (int i = 0; i < kPer; i++) d[threadIdx.x + i * kTileThreads] = v[i];
    } else {
      for (int j = threadIdx.x; j < cnt; j += kTileThreads) win[j] = cin[base + j];
    }
    __syncthreads();
    // Each wavefront's next chunk is loaded before the current one is summed
    // and stored, so its wait does not include those stores (vector memory
    // operations complete in issue order).  Two load buffers alternate, so no
    // copy between them waits early.  The load after the range's last chunk
    // repeats that chunk and is not summed.
    int64_t cb = c + wave;
    if (cb < wend) {
      ChunkLoad ca = load_chunk(t, cb, lane);
      chunk_ready(ca);
      for (;;) {
        const ChunkLoad cn = load_chunk(t, min(cb + kWaves, wend - 1), lane);
        tile_chunk(t, win, ca, lane, stage);
        cb += kWaves;
        if (cb >= wend) break;
        ca = load_chunk(t, min(cb + kWaves, wend - 1), lane);
        tile_chunk(t, win, cn, lane, stage);
        cb += kWaves;
        if (cb >= wend) break;
      }
    }
    c = wend;
  }
}

// Compensated merge of the region's partials reg[ix[0..cnt)] in order; the
// offsets are loaded kMergeAhead at a time, all before their LDS reads.
constexpr int kMergeAhead = 8;
__device__ __forceinline__ Comp merge_list(const float* reg, const uint16_t* __restrict__ ix, int cnt) {
  Comp acc{0.0f, 0.0f};
  for (int k = 0; k < cnt; k += kMergeAhead) {
    uint16_t q[kMergeAhead];
#pragma unroll
    for (int j = 0; j < kMergeAhead; j++) q[j] = k + j < cnt ? ix[k + j] : 0;
#pragma unroll
    for (int j = 0; j < kMergeAhead; j++) {
      const float v = reg[q[j]];
      if (k + j < cnt) acc.add(v);
    }
  }
  return acc;
}

constexpr int kSegBatch = kRowThreads;  // segments staged per round
constexpr int kXcds = 8;                 // MI355X: 8 XCDs, each with its own L2
constexpr int kRegionPer = kRowSlots / kRowThreads;  // region entries per thread
constexpr int kGroupShift = 5;           // region entries per search group: 32
constexpr int kGroups = kRowSlots >> kGroupShift;
static_assert(kSegBatch <= 32767, "segment numbers are stored as int16");

// Row pass of the tiled mode: persistent workgroups take row blocks in
// turn.  A block's region (its partials, window order) is gathered into LDS
// from its segments: every thread loads its region entries (all loads in
// flight before the LDS stores), finding each entry's segment by binary
// search over the segments' region offsets, between the segments that hold
// the first entries of its 32-entry group and of the next group.  A one-row block merges its
// region with its threads striding it in order, then a fixed tree; in a
// multi-row block every thread merges one row's partials in window order.
// Rows without in-edges (the tail) only finish.
__global__ __launch_bounds__(kRowThreads, kRowGroupsPerCU * kRowThreads / 256) void k_rows(PrArgs a, TileArgs t, float* __restrict__ cout,
                                                     float* __restrict__ score) {
  __shared__ float reg[kRowSlots];
  __shared__ int32_t soff[kSegBatch + 1];
  __shared__ int32_t sstart[kSegBatch];
  __shared__ int16_t gseg[kGroups + 1];  // segment of each group's first entry
  __shared__ float2 wred[kRowThreads / 64];
  __shared__ double red[kRowThreads / 64];
  if (a.ctrl->pad) return;
  double err = 0;
  const int lane = lane_id();
  const int wave = threadIdx.x >> 6;
  const int k = static_cast<int>(threadIdx.x);
  // XCD-aware order: workgroups are dealt round-robin to the kXcds XCDs, so
  // workgroup g runs on XCD g % kXcds.  Blocks go out in groups of W
  // consecutive blocks (W = workgroups per XCD), group j to XCD j % kXcds,
  // so in each round one XCD's workgroups take W neighbouring blocks, whose
  // segments share lines of the partial array, and the XCDs alternate
  // groups along the whole block range.
  const int64_t W = gridDim.x % kXcds == 0 ? gridDim.x / kXcds : 0;
  const int64_t xcd = blockIdx.x % kXcds, lw = blockIdx.x / kXcds;
  for (int64_t i = 0;; i++) {
    const int64_t b = W ? (xcd + kXcds * i) * W + lw : blockIdx.x + i * gridDim.x;
    if (b >= t.n_blocks) break;
    const int32_t r0 = t.brow[b], r1 = t.brow[b + 1];
    const int64_t s0 = t.bseg[b], s1 = t.bseg[b + 1];
    const int32_t size = t.bsize[b];
    // Gather the region, kSegBatch segments per round.
    for (int64_t sb = s0; sb < s1; sb += kSegBatch) {
      const int ns = static_cast<int>(min<int64_t>(kSegBatch, s1 - sb));
      if (k < ns) {
        sstart[k] = t.seg_start[sb + k];
        soff[k] = t.seg_off[sb + k];
      }
      if (k == 0) soff[ns] = sb + ns < s1 ? t.seg_off[sb + ns] : size;
      __syncthreads();
      const int lo_e = soff[0], hi_e = soff[ns];
      const int ngroups = (hi_e - lo_e + (1 << kGroupShift) - 1) >> kGroupShift;
      if (k < ns) {
        // Segments are not empty; group g's first entry lo_e + 32 g lies in
        // exactly one of them.
        const int g0 = (soff[k] - lo_e + (1 << kGroupShift) - 1) >> kGroupShift;
        const int g1 = (soff[k + 1] - lo_e + (1 << kGroupShift) - 1) >> kGroupShift;
        for (int g = g0; g < g1; g++) gseg[g] = static_cast<int16_t>(k);
      }
      __syncthreads();
      float v[kRegionPer];
#pragma unroll
      for (int i = 0; i < kRegionPer; i++) {
        const int e = lo_e + k + i * kRowThreads;
        if (e < hi_e) {
          // The last segment with soff <= e, between the segments of this
          // group's first entry and of the next group's.
          const int g = (e - lo_e) >> kGroupShift;
          int lo = gseg[g], hi = g + 1 < ngroups ? gseg[g + 1] + 1 : ns;
          while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (soff[mid] <= e) lo = mid; else hi = mid;
          }
          v[i] = t.part[sstart[lo] + (e - soff[lo])];
        }
      }
#pragma unroll
      for (int i = 0; i < kRegionPer; i++) {
        const int e = lo_e + k + i * kRowThreads;
        if (e < hi_e) reg[e] = v[i];
      }
      __syncthreads();
    }
    if (r1 - r0 == 1) {
      FusedAcc<float> acc;
      for (int p = k; p < size; p += kRowThreads) acc.add(reg[p]);
      acc.reduce<64>(lane);
      if (lane == 0) wred[wave] = make_float2(acc.c.s, acc.c.c);
      __syncthreads();
      if (k == 0) {
        Comp tot = {wred[0].x, wred[0].y};
        for (int w = 1; w < kRowThreads / 64; w++) tot.merge(wred[w].x, wred[w].y);
        err += finish_f32(a, r0, tot.value(), score, cout);
      }
      __syncthreads();
      continue;
    }
    for (int32_t r = r0 + k; r < r1; r += kRowThreads) {
      // The row's old score and out-degree load beside its list bounds,
      // ahead of the merge.
      const int32_t i0 = t.istart[r], i1 = t.istart[r + 1];
      const float old = score[r];
      const int64_t deg = out_deg(a, r);
      const Comp acc = merge_list(reg, t.idx + i0, i1 - i0);
      const float nw = a.prm->base_f + a.prm->damp_f * acc.value();
      score[r] = nw;
      cout[r] = nw / static_cast<float>(deg);
      err += static_cast<double>(fabsf(nw - old));
    }
    __syncthreads();  // LDS readers done before the next block's gather
  }
  for (int64_t u = a.zero_begin + int64_t(blockIdx.x) * kRowThreads + threadIdx.x; u < a.nloc;
       u += int64_t(gridDim.x) * kRowThreads)
    err += finish_f32(a, u, 0.0f, score, cout);
  const double tt = block_err_sum<kRowThreads>(err, red);
  if (threadIdx.x == 0) a.err_part[blockIdx.x] = tt;
}

// Merges each split row's segment partials in segment order and finishes it.
__global__ __launch_bounds__(kThreads) void k_kahan_super(PrArgs a, float* __restrict__ cout,
                                                          float* __restrict__ score) {
  __shared__ double red[kThreads / 64];
  if (a.ctrl->pad) return;
  double err = 0;
  const int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  if (i < a.n_super) {
    const PrSuper sp = a.supers[i];
    const double2 p0 = a.partial[sp.first];
    Comp acc{static_cast<float>(p0.x), static_cast<float>(p0.y)};
    for (int j = 1; j < sp.count; j++) {
      const double2 p = a.partial[sp.first + j];
      acc.merge(static_cast<float>(p.x), static_cast<float>(p.y));
    }
    err = finish_f32(a, sp.v, acc.value(), score, cout);
  }
  double t = block_err_sum(err, red);
  if (threadIdx.x == 0) a.err_part[a.main_blocks + blockIdx.x] = t;
}

__global__ __launch_bounds__(kThreads) void k_f64_super(PrArgs a, double* __restrict__ cout,
                                                        double* __restrict__ score) {
  __shared__ double red[kThreads / 64];
  if (a.ctrl->pad) return;
  double err = 0;
  const int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  if (i < a.n_super) {
    const PrSuper sp = a.supers[i];
    double acc = 0;
    for (int j = 0; j < sp.count; j++) acc += a.partial[sp.first + j].x;
    err = finish_f64(a, sp.v, acc, score, cout);
  }
  double t = block_err_sum(err, red);
  if (threadIdx.x == 0) a.err_part[a.main_blocks + blockIdx.x] = t;
}

// ---- FP32_KAHAN on a PE block: propagation layout, exact sums ---------------
//
// Pass 1 (k_bprop) gathers every in-edge's contribution from an LDS copy of
// its source's window and writes it to the edge's place in the bucket-major
// array; pass 2 (k_bsum) sums each bucket's rows.  The sums are exact: a
// contribution c enters as the 128-bit two's complement integer
// c * 2^kFxShift (exact for |c| >= 2^-57, truncated below 2^-kFxShift), so
// the order of the additions does not matter and the LDS accumulators take
// plain integer atomics; each row's sum is rounded to FP32 once.  Row sums
// must stay below 2^47 in magnitude (PageRank contributions are in [0, 1]).

constexpr int kBPropThreads = 1024;
constexpr int kBSumThreads = 1024;
constexpr int kFxShift = 80;

struct BpArgs {
  const uint16_t* src;
  const int64_t* wstart;
  const int32_t* wlen;
  const int64_t* wseg;
  const int32_t* seg_d;
  const int64_t* wgroup;
  const BlockGroup* groups;
  const uint16_t* brow;
  const FineRow* rows;
  const BlockUnit* units;
  const BlockSplit* splits;
  float* val;
  float* spare;     // val[m]: the stores of lanes past a window's end
  long long* part;  // (lo, hi) per partial slot
  int32_t nwin;
  int32_t wparts;   // workgroups that share a window
  int64_t n_units, n_splits;
};

// c * 2^kFxShift as a 128-bit two's complement integer (lo, hi).
__device__ __forceinline__ void fx_of(float c, unsigned long long& lo, long long& hi) {
  const unsigned bits = __float_as_uint(c);
  const int e = static_cast<int>((bits >> 23) & 0xFFu);
  const unsigned long long m = (bits & 0x7FFFFFu) | 0x800000u;
  lo = 0;
  hi = 0;
  if (e == 0) return;  // zero or subnormal: below 2^-126
  const int sh = e - 150 + kFxShift;  // |c| = m * 2^(e - 150)
  if (sh <= -24) return;
  if (sh < 0) {
    lo = m >> (-sh);
  } else if (sh < 64) {
    lo = m << sh;
    hi = sh > 40 ? static_cast<long long>(m >> (64 - sh)) : 0;
  } else {
    hi = static_cast<long long>(m << (sh - 64));
  }
  if (bits >> 31) {
    lo = ~lo + 1;
    hi = ~hi + (lo == 0 ? 1 : 0);
  }
}

__device__ __forceinline__ void fx_add(unsigned long long& lo, long long& hi, unsigned long long xlo, long long xhi) {
  const unsigned long long s = lo + xlo;
  hi += xhi + (s < lo ? 1 : 0);
  lo = s;
}

// The FP32 rounding (to nearest) of the 128-bit integer (lo, hi) * 2^-kFxShift:
// the top 64 significant bits, with any lower bit set folded into the last
// (sticky) bit, convert to FP32 with one rounding; the scaling by a power of
// two is exact.
__device__ __forceinline__ float fx_value(unsigned long long lo, long long hi) {
  const bool neg = hi < 0;
  if (neg) {
    lo = ~lo + 1;
    hi = ~hi + (lo == 0 ? 1 : 0);
  }
  const unsigned long long uh = static_cast<unsigned long long>(hi);
  float f;
  if (uh == 0) {
    f = ldexpf(static_cast<float>(lo), -kFxShift);
  } else {
    const int lz = __clzll(static_cast<long long>(uh));
    const unsigned long long top = lz ? (uh << lz) | (lo >> (64 - lz)) : uh;
    const unsigned long long rest = lz ? lo << lz : lo;
    f = ldexpf(static_cast<float>(top | (rest != 0 ? 1ull : 0ull)), 64 - lz - kFxShift);
  }
  return neg ? -f : f;
}

// Pass 1: persistent workgroups take windows in turn, or parts of one where
// there are fewer windows than CUs.  A window's contributions and segment
// table go to LDS.  A wavefront takes kBPer groups of 64 consecutive edges at
// a time, lane l the l-th edge of each group, so every store instruction
// writes 64 consecutive destinations inside a segment (segments average tens
// of edges).  A lane's segment is the group's first plus the segment starts
// up to its edge, counted in the group's mask.  The next round's source
// offsets and masks are loaded before this round's stores.
__global__ __launch_bounds__(kBPropThreads) void k_bprop(BpArgs b, const float* __restrict__ cin, int64_t n_gather,
                                                         PrHead head) {
  __shared__ float win[kBWin];
  __shared__ int32_t sd[kBSegMax];
  if (head.prm && blockIdx.x == 0 && threadIdx.x == 0) write_head(head);  // for the kernels that follow
  const int lane = lane_id();
  const int wv = threadIdx.x >> 6;
  constexpr int kRound = 64 * kBPer;                         // edges per wavefront round
  constexpr int kStride = (kBPropThreads / 64) * kRound;     // edges per workgroup round
  for (int32_t item = blockIdx.x; item < b.nwin * b.wparts; item += gridDim.x) {
    const int32_t w = item % b.nwin, part = item / b.nwin;
    const int64_t base = int64_t(w) * kBWin;
    const int cnt = static_cast<int>(min<int64_t>(kBWin, n_gather - base));
    const int64_t s0 = b.wseg[w];
    const int ns = static_cast<int>(b.wseg[w + 1] - s0);
    // This part's edges [begin, len) of the window (whole rounds).
    const int per = (b.wlen[w] + b.wparts * kStride - 1) / (b.wparts * kStride) * kStride;
    const int begin = part * per;
    const int len = min(b.wlen[w], begin + per);
    if (begin >= len) continue;
    const uint16_t* src = b.src + b.wstart[w];
    __syncthreads();  // the previous window's readers are done
    if (cnt == kBWin && (reinterpret_cast<uintptr_t>(cin) & 15) == 0) {
      const float4* s4 = reinterpret_cast<const float4*>(cin + base);
      float4* d4 = reinterpret_cast<float4*>(win);
      constexpr int kPer = kBWin / 4 / kBPropThreads;
      float4 v[kPer];
#pragma unroll
      for (int i = 0; i < kPer; i++) v[i] = s4[threadIdx.x + i * kBPropThreads];
#pragma unroll
      for (int i = 0; i < kPer; i++) d4[threadIdx.x + i * kBPropThreads] = v[i];
    } else {
      for (int j = threadIdx.x; j < cnt; j += kBPropThreads) win[j] = cin[base + j];
    }
    for (int k = threadIdx.x; k < ns; k += kBPropThreads) sd[k] = b.seg_d[s0 + k];
    const BlockGroup* groups = b.groups + b.wgroup[w];
    const int last_group = (b.wlen[w] - 1) >> 6;
    __syncthreads();
    // A wavefront's next round of offsets and masks loads at the start of the
    // current round, into one of two buffers that alternate (no copy, which
    // would wait).  Vector loads and stores complete in issue order; with
    // unconditional loads (index clamped into the window) and stores, every
    // path issues the same count, so the next round waits for its offsets
    // with a count that leaves this round's stores in flight.
    struct Round {
      uint32_t q[kBPer];
      BlockGroup g;  // lane k: the round's k-th group
    };
    auto load_round = [&](int c, Round& r) {
#pragma unroll
      for (int k = 0; k < kBPer; k++) r.q[k] = src[min(c + lane + 64 * k, len - 1)];
      r.g = groups[min((c >> 6) + (lane & (kBPer - 1)), last_group)];
    };
    auto round = [&](int c0, const Round& r, Round& next) {
      load_round(c0 + kStride, next);
      // Every lane stores kBPer times (lanes past the part's end into the
      // spare slot), so every path issues the same number of stores.
#pragma unroll
      for (int k = 0; k < kBPer; k++) {
        const int i = c0 + lane + 64 * k;
        const unsigned lo = __builtin_amdgcn_readlane(static_cast<unsigned>(r.g.starts), k);
        const unsigned hi = __builtin_amdgcn_readlane(static_cast<unsigned>(r.g.starts >> 32), k);
        const int sg = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, __builtin_amdgcn_readlane(r.g.first, k)));
        float* dst = b.val + int64_t(sd[min(sg, ns - 1)]) + i;
        *(i < len ? dst : b.spare) = win[r.q[k]];
      }
    };
    int c0 = begin + wv * kRound;
    if (c0 < len) {
      Round ra, rb;
      load_round(c0, ra);
#pragma unroll
      for (int k = 0; k < kBPer; k++) __asm__ volatile("" ::"v"(ra.q[k]));
      __asm__ volatile("" ::"v"(ra.g.first));
      for (;;) {
        round(c0, ra, rb);
        c0 += kStride;
        if (c0 >= len) break;
        round(c0, rb, ra);
        c0 += kStride;
        if (c0 >= len) break;
      }
    }
  }
}

// A unit of one row, by the workgroup: summed in registers.
constexpr int kBSumUnroll = 8;
__device__ __forceinline__ void one_row_unit(const PrArgs& a, const BpArgs& b, const BlockUnit& U,
                                             unsigned long long* rlo, long long* rhi, double& err, float* cout,
                                             float* score) {
  constexpr int64_t kStep = int64_t(kBSumThreads) * kBSumUnroll;
  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int wave = tid >> 6;
  unsigned long long lo = 0;
  long long hi = 0;
  for (int64_t e = U.e0 + tid; e < U.e1; e += kStep) {
    float v[kBSumUnroll];
#pragma unroll
    for (int j = 0; j < kBSumUnroll; j++) v[j] = e + j * kBSumThreads < U.e1 ? b.val[e + j * kBSumThreads] : 0.0f;
#pragma unroll
    for (int j = 0; j < kBSumUnroll; j++) {
      unsigned long long xl;
      long long xh;
      fx_of(v[j], xl, xh);
      fx_add(lo, hi, xl, xh);
    }
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    const unsigned long long ol = __shfl_xor(lo, d);
    const long long oh = __shfl_xor(hi, d);
    fx_add(lo, hi, ol, oh);
  }
  if (lane == 0) {
    rlo[wave] = lo;
    rhi[wave] = hi;
  }
  __syncthreads();
  if (tid == 0) {
    unsigned long long tl = 0;
    long long th = 0;
    for (int w = 0; w < kBSumThreads / 64; w++) fx_add(tl, th, rlo[w], rhi[w]);
    if (U.slot >= 0) {
      b.part[2 * int64_t(U.slot)] = static_cast<long long>(tl);
      b.part[2 * int64_t(U.slot) + 1] = th;
    } else {
      err += finish_f32(a, U.row0, fx_value(tl, th), score, cout);
    }
  }
  __syncthreads();
}

template <int kCtrl, int kRowMask>
__device__ __forceinline__ long long dpp_move64(long long x) {
  const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(x), kCtrl, kRowMask, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(x >> 32), kCtrl, kRowMask, 0xf, true);
  return (static_cast<long long>(hi) << 32) | static_cast<unsigned int>(lo);
}

// Sum over groups of kLanes lanes (1, 8 or 64), valid in a group's last lane.
template <int kCtrl, int kRowMask, typename T>
__device__ __forceinline__ T dpp_moved(T x) {
  long long b;
  __builtin_memcpy(&b, &x, 8);
  b = dpp_move64<kCtrl, kRowMask>(b);
  __builtin_memcpy(&x, &b, 8);
  return x;
}
template <int kLanes, typename T>
__device__ __forceinline__ T group_sum(T x) {
  if (kLanes > 1) {
    x += dpp_moved<0x111, 0xf>(x);  // row_shr:1
    x += dpp_moved<0x112, 0xf>(x);  // row_shr:2
    x += dpp_moved<0x114, 0xf>(x);  // row_shr:4
  }
  if (kLanes == 64) {
    x += dpp_moved<0x118, 0xf>(x);  // row_shr:8
    x += dpp_moved<0x142, 0xa>(x);  // row_bcast:15 into rows 1 and 3
    x += dpp_moved<0x143, 0xc>(x);  // row_bcast:31 into rows 2 and 3
  }
  return x;
}

// Exact sums of contributions (multiples of 2^-kFxShift), as two doubles
// where every |c| of the unit is 0 or in [2^-57, 1/4] (FineHalves), else as
// 128-bit integers (FineFixed).
//
// Halves: c = h + l with h the nearest multiple of 2^-40 and l a multiple of
// 2^-80 of at most 2^-41.  A unit has at most 2^14 values, so sums of h stay
// at most 2^52 units and sums of l at most 2^53: neither is ever rounded, in
// any order, and h + l is the exact sum.  Five double additions a value where
// the integers take some twenty instructions.
constexpr float kHalvesMin = 0x1p-57f, kHalvesMax = 0.25f;
static_assert(kFineEdges <= 1 << 14, "exact sums of halves");

struct FineHalves {
  double h = 0.0, l = 0.0;
  __device__ __forceinline__ void add(float c) {
    constexpr double kRound = 0x1.8p12;  // adding it rounds to multiples of 2^-40
    const double d = static_cast<double>(c);
    const double t = (d + kRound) - kRound;
    h += t;
    l += d - t;
  }
  template <int kLanes>
  __device__ __forceinline__ void reduce() {
    h = group_sum<kLanes>(h);
    l = group_sum<kLanes>(l);
  }
  // To a row's accumulator in LDS (two words, zeroed), from any wavefront.
  __device__ __forceinline__ void add_to(unsigned long long* a, unsigned long long* b) const {
    atomicAdd(reinterpret_cast<double*>(a), h);
    atomicAdd(reinterpret_cast<double*>(b), l);
  }
  static __device__ __forceinline__ FineHalves of(unsigned long long a, unsigned long long b) {
    FineHalves r;
    __builtin_memcpy(&r.h, &a, 8);
    __builtin_memcpy(&r.l, &b, 8);
    return r;
  }
  // h + l rounded once to FP32: rounded to odd in double (which keeps, in its
  // last bit, that something was cut off), then to nearest.
  __device__ __forceinline__ float value() const {
    const double s = h + l;
    const double bb = s - h;
    const double e = (h - (s - bb)) + (l - bb);
    long long bits = __double_as_longlong(s);
    if (e != 0.0 && (bits & 1) == 0) bits += (e > 0.0) == (s > 0.0) ? 1 : -1;
    return static_cast<float>(__longlong_as_double(bits));
  }
};

struct FineFixed {
  unsigned long long lo = 0;
  long long hi = 0;
  __device__ __forceinline__ void add(float c) {
    unsigned long long xl;
    long long xh;
    fx_of(c, xl, xh);
    fx_add(lo, hi, xl, xh);
  }
  // Three limbs of 48 bits, whose sums over lanes carry nothing.
  template <int kLanes>
  __device__ __forceinline__ void reduce() {
    if (kLanes == 1) return;
    constexpr unsigned long long kMask = (1ull << 48) - 1;
    const long long l0 = group_sum<kLanes>(static_cast<long long>(lo & kMask));
    const long long l1 =
        group_sum<kLanes>(static_cast<long long>(((lo >> 48) | (static_cast<unsigned long long>(hi) << 16)) & kMask));
    const long long l2 = group_sum<kLanes>(hi >> 32);
    lo = static_cast<unsigned long long>(l0);
    hi = l2 << 32;
    fx_add(lo, hi, static_cast<unsigned long long>(l1) << 48, l1 >> 16);
  }
  __device__ __forceinline__ void add_to(unsigned long long* a, unsigned long long* b) const {
    const unsigned long long old = atomicAdd(a, lo);
    atomicAdd(b, static_cast<unsigned long long>(hi) + (old + lo < old ? 1 : 0));
  }
  static __device__ __forceinline__ FineFixed of(unsigned long long a, unsigned long long b) {
    FineFixed r;
    r.lo = a;
    r.hi = static_cast<long long>(b);
    return r;
  }
  __device__ __forceinline__ float value() const { return fx_value(lo, hi); }
};

// The exact sum of places [begin, end), by kLanes lanes of which this is the
// sub-th, kFineAhead reads ahead; valid in the last one.
constexpr int kFineAhead = 4;
template <typename Acc, int kLanes>
__device__ __forceinline__ Acc fine_sum(const float* place, int begin, int end, int sub) {
  Acc acc;
  for (int k = begin + sub; k < end; k += kLanes * kFineAhead) {
    float x[kFineAhead];
#pragma unroll
    for (int j = 0; j < kFineAhead; j++) x[j] = place[min(k + j * kLanes, end - 1)];
#pragma unroll
    for (int j = 0; j < kFineAhead; j++) acc.add(k + j * kLanes < end ? x[j] : 0.0f);
  }
  acc.template reduce<kLanes>();
  return acc;
}

constexpr int kFineLongs = kFineEdges / kFineLong;
static_assert(kFineLongs <= 64, "a lane per long row");

struct FineLds {
  float place[kFineEdges];
  float sums[kFineRows];
  unsigned long long la[kFineLongs], lb[kFineLongs];  // the long rows' accumulators
  int fixed;  // the unit last found with a contribution outside the halves' range
};

// The row sums of a unit whose contributions are in place.
template <typename Acc>
__device__ __forceinline__ void fine_rows(const BlockUnit& U, const FineRow* rows, FineLds& L) {
  constexpr int kWaves = kBSumThreads / 64;
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int short0 = U.nlong + U.nmid;
  if (U.nlong > 0) {
    // The long rows hold places [0, end): this wavefront's share, row by row.
    const FineRow mine = rows[min(lane, U.nlong - 1)];
    const int end = __builtin_amdgcn_readlane(mine.start + mine.len, U.nlong - 1);
    const int per = (end + kWaves - 1) / kWaves;
    const int p1 = min(end, (wave + 1) * per);
    int p = wave * per;
    int i = __popcll(__ballot(lane < U.nlong && mine.start <= p)) - 1;
    while (p < p1) {
      const int stop = min(p1, __builtin_amdgcn_readlane(mine.start + mine.len, i));
      const Acc acc = fine_sum<Acc, 64>(L.place, p, stop, lane);
      if (lane == 63) acc.add_to(&L.la[i], &L.lb[i]);
      p = stop;
      i++;
    }
  }
  for (int i0 = U.nlong + wave * 8; i0 < short0; i0 += kWaves * 8) {
    const int i = i0 + (lane >> 3);
    const FineRow r = rows[min(i, short0 - 1)];
    const Acc acc = fine_sum<Acc, 8>(L.place, r.start, r.start + r.len, lane & 7);
    if (i < short0 && (lane & 7) == 7) L.sums[r.row] = acc.value();
  }
  for (int i = short0 + threadIdx.x; i < U.nrows; i += kBSumThreads) {
    const FineRow r = rows[i];
    L.sums[r.row] = fine_sum<Acc, 1>(L.place, r.start, r.start + r.len, 0).value();
  }
  if (U.nlong > 0) {
    __syncthreads();
    const int i = threadIdx.x;
    if (i < U.nlong) L.sums[rows[i].row] = Acc::of(L.la[i], L.lb[i]).value();
  }
}

// Pass 2, fine buckets: a unit's contributions go to their places in LDS,
// rows by length, and each row's run is summed in registers: short rows by a
// thread, middling ones by eight lanes, and the long ones' places are shared
// out evenly, each wavefront adding what it has of a row to the row's
// accumulator; then the rows finish, in order.  One LDS write and one read
// per edge where the coarse pass has 64-bit atomics.
__global__ __launch_bounds__(kBSumThreads, 8) void k_bfine(PrArgs a, BpArgs b, float* __restrict__ cout,
                                                           float* __restrict__ score) {
  __shared__ FineLds L;
  __shared__ unsigned long long rlo[kBSumThreads / 64];
  __shared__ long long rhi[kBSumThreads / 64];
  __shared__ double red[kBSumThreads / 64];
  if (a.ctrl->pad) return;
  double err = 0;
  const int tid = threadIdx.x;
  constexpr int kPer = kFineEdges / kBSumThreads;
  if (tid == 0) L.fixed = -1;  // no unit
  __syncthreads();
  for (int u = blockIdx.x; u < b.n_units; u += gridDim.x) {
    const BlockUnit U = b.units[u];
    if (U.nrows == 1) {
      one_row_unit(a, b, U, rlo, rhi, err, cout, score);
      continue;
    }
    const int n = static_cast<int>(U.e1 - U.e0);
    if (n > 0) {
      // All loads first (past the end the last edge again), then the stores.
      float v[kPer];
      int at[kPer];
#pragma unroll
      for (int j = 0; j < kPer; j++) {
        const int64_t e = U.e0 + min(tid + j * kBSumThreads, n - 1);
        v[j] = b.val[e];
        at[j] = b.brow[e];
      }
      bool halves = true;
#pragma unroll
      for (int j = 0; j < kPer; j++) {
        L.place[at[j]] = v[j];
        const float c = fabsf(v[j]);
        halves = halves && (c == 0.0f || (c >= kHalvesMin && c <= kHalvesMax));
      }
      if (!halves) L.fixed = u;
    }
    if (tid < kFineLongs) L.la[tid] = L.lb[tid] = 0;
    __syncthreads();
    if (L.fixed != u)
      fine_rows<FineHalves>(U, b.rows + U.row0, L);
    else
      fine_rows<FineFixed>(U, b.rows + U.row0, L);
    __syncthreads();
    for (int r = tid; r < U.nrows; r += kBSumThreads) err += finish_f32(a, int64_t(U.row0) + r, L.sums[r], score, cout);
  }
  const double t = block_err_sum<kBSumThreads>(err, red);
  if (threadIdx.x == 0) a.err_part[blockIdx.x] = t;
}

// Pass 2, coarse buckets: persistent workgroups take units in turn.  A bucket
// of several rows accumulates in LDS (128-bit integer per row: the low word by a
// 64-bit atomic add, its carry and the high word by a second); a one-row
// unit in registers, reduced over the workgroup.  Rows finish here, except
// the parts of a one-row bucket beyond kBEdges edges, whose sums go to
// partial slots for k_bsplit.
__global__ __launch_bounds__(kBSumThreads) void k_bsum(PrArgs a, BpArgs b, float* __restrict__ cout,
                                                       float* __restrict__ score) {
  __shared__ unsigned long long alo[kBRows];
  __shared__ unsigned long long ahi[kBRows];
  __shared__ unsigned long long rlo[kBSumThreads / 64];
  __shared__ long long rhi[kBSumThreads / 64];
  __shared__ double red[kBSumThreads / 64];
  if (a.ctrl->pad) return;
  double err = 0;
  const int tid = threadIdx.x;
  constexpr int64_t kStep = int64_t(kBSumThreads) * kBSumUnroll;
  for (int64_t u = blockIdx.x; u < b.n_units; u += gridDim.x) {
    const BlockUnit U = b.units[u];
    if (U.nrows == 1) {
      one_row_unit(a, b, U, rlo, rhi, err, cout, score);
      continue;
    }
    for (int r = tid; r < U.nrows; r += kBSumThreads) {
      alo[r] = 0;
      ahi[r] = 0;
    }
    __syncthreads();
    // Each round's loads are issued before the previous round's atomics.
    float v[kBSumUnroll];
    int r[kBSumUnroll];
    int64_t e = U.e0 + tid;
#pragma unroll
    for (int j = 0; j < kBSumUnroll; j++) {
      const int64_t k = e + j * kBSumThreads;
      v[j] = k < U.e1 ? b.val[k] : 0.0f;
      r[j] = k < U.e1 ? b.brow[k] : 0;
    }
    for (; e < U.e1; e += kStep) {
      float vn[kBSumUnroll];
      int rn[kBSumUnroll];
#pragma unroll
      for (int j = 0; j < kBSumUnroll; j++) {
        const int64_t k = e + kStep + j * kBSumThreads;
        vn[j] = k < U.e1 ? b.val[k] : 0.0f;
        rn[j] = k < U.e1 ? b.brow[k] : 0;
      }
#pragma unroll
      for (int j = 0; j < kBSumUnroll; j++) {
        unsigned long long xl;
        long long xh;
        fx_of(v[j], xl, xh);
        if (xl | static_cast<unsigned long long>(xh)) {
          const unsigned long long old = atomicAdd(&alo[r[j]], xl);
          const long long c = xh + (old + xl < old ? 1 : 0);
          if (c) atomicAdd(&ahi[r[j]], static_cast<unsigned long long>(c));
        }
      }
#pragma unroll
      for (int j = 0; j < kBSumUnroll; j++) {
        v[j] = vn[j];
        r[j] = rn[j];
      }
    }
    __syncthreads();
    for (int rr = tid; rr < U.nrows; rr += kBSumThreads)
      err += finish_f32(a, U.row0 + rr, fx_value(alo[rr], static_cast<long long>(ahi[rr])), score, cout);
    __syncthreads();
  }
  const double t = block_err_sum<kBSumThreads>(err, red);
  if (threadIdx.x == 0) a.err_part[blockIdx.x] = t;
}

// The last iteration's error (the others' are reduced by the kernel that
// follows them, pr_begin), by one workgroup; partial `own` is `mine`.
__device__ __forceinline__ void reduce_error(const PrArgs& a, int own, double mine, double* red) {
  PrCtrl* c = a.ctrl;
  const double t = error_sum<kThreads>(a.err_part, a.main_blocks + a.super_blocks, own, mine, red);
  if (threadIdx.x == 0) {
    const unsigned it = c->ticket;
    c->err = t;
    if (it < DMM_MAX_PR_ITERS) a.err_trace[it] = t;
    if (a.err_out) *a.err_out = t;
    c->ticket = it + 1;
    if (t < a.prm->eps) c->pad = 1;
  }
}

// The one-row buckets in parts: each row's partial sums (exact) in slot order,
// then the row finishes.  With one workgroup (up to kThreads split rows) also
// the reduction of the error, 4 us of a launch less.
__global__ __launch_bounds__(kThreads) void k_bsplit(PrArgs a, BpArgs b, float* __restrict__ cout,
                                                     float* __restrict__ score) {
  __shared__ double red[kThreads / 64];
  __shared__ double mine;
  double err = 0;
  const int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  if (i < b.n_splits) {
    const BlockSplit sp = b.splits[i];
    unsigned long long lo = 0;
    long long hi = 0;
    for (int j = 0; j < sp.count; j++)
      fx_add(lo, hi, static_cast<unsigned long long>(b.part[2 * int64_t(sp.first + j)]),
             b.part[2 * int64_t(sp.first + j) + 1]);
    err = finish_f32(a, sp.row, fx_value(lo, hi), score, cout);
  }
  const double t = block_err_sum(err, red);
  if (gridDim.x > 1) {
    if (threadIdx.x == 0) a.err_part[a.main_blocks + blockIdx.x] = t;
    return;
  }
  if (threadIdx.x == 0) mine = t;
  __syncthreads();
  reduce_error(a, a.main_blocks, mine, red);
}

// ---- iteration bookkeeping --------------------------------------------------

__global__ __launch_bounds__(kThreads) void k_reduce(PrArgs a) {
  __shared__ double red[kThreads / 64];
  if (a.ctrl->pad) return;
  reduce_error(a, -1, 0.0, red);
}

__global__ __launch_bounds__(kThreads) void k_init_f32(PrArgs a, float* score, float* contrib) {
  const int64_t gtid = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  const int64_t gsize = int64_t(gridDim.x) * kThreads;
  const float init = a.prm->init_f;
  for (int64_t u = gtid; u < a.nloc; u += gsize) {
    score[u] = init;
    contrib[u] = init / static_cast<float>(out_deg(a, u));  // src/pr.cc:52-53
  }
  if (gtid == 0) {
    a.ctrl->pad = 0;
    a.ctrl->ticket = 0;
    a.ctrl->err = 0;
  }
}

__global__ __launch_bounds__(kThreads) void k_init_f64(PrArgs a, double* score, double* contrib) {
  const int64_t gtid = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  const int64_t gsize = int64_t(gridDim.x) * kThreads;
  const double init = a.prm->init_d;
  for (int64_t u = gtid; u < a.nloc; u += gsize) {
    score[u] = init;
    contrib[u] = init / static_cast<double>(out_deg(a, u));
  }
  if (gtid == 0) {
    a.ctrl->pad = 0;
    a.ctrl->ticket = 0;
    a.ctrl->err = 0;
  }
}

__global__ void k_reset_ctrl(PrCtrl* c) {
  c->pad = 0;
  c->ticket = 0;
  c->err = 0;
}

PrArgs make_args(dmm_ctx* ctx) {
  PrArgs a;
  a.in_off = ctx->d_in_off;
  a.in_nbr = ctx->d_in_nbr;
  a.out_off = ctx->d_out_off;
  a.heavy = ctx->d_heavy;
  a.items = static_cast<const PrItem*>(ctx->d_items);
  a.supers = static_cast<const PrSuper*>(ctx->d_supers);
  a.partial = static_cast<double2*>(ctx->d_partial);
  a.nloc = ctx->nloc;
  a.n_heavy = ctx->n_heavy;
  a.n_items = ctx->n_items;
  a.n_super = ctx->n_super;
  a.heavy_threshold = ctx->heavy_threshold;
  a.err_part = ctx->d_err_part;
  a.sitems = static_cast<const SerialItem*>(ctx->d_sitems);
  a.sstart = ctx->d_sstart;
  // In the degree order the first vertices receive most gathers; in another
  // order they do only if they are most of the vertices.
  a.serial_hub = ctx->relabeled || ctx->n <= 2 * kSerialHub ? static_cast<int>(std::min<int64_t>(kSerialHub, ctx->n)) : 0;
  a.super_blocks = pr_super_blocks(ctx);
  a.main_blocks = 0;
  a.n_gather = ctx->n;
  a.light_begin = ctx->pr_light_begin;
  a.light_end = ctx->pr_light_end;
  a.zero_begin = ctx->pr_zero_begin;
  a.ctrl = ctx->d_prctrl;
  a.err_trace = ctx->d_err_trace;
  a.err_out = nullptr;
  a.prm = reinterpret_cast<const PrParams*>(ctx->d_prparams);
  return a;
}

// Error partials an iteration of `mode` writes (block: a PE block's iteration
// from the global contributions).
int pr_error_parts(dmm_ctx* ctx, int mode, bool block) {
  if (mode == DMM_PR_FP32_SERIAL) return pr_serial_blocks(ctx);
  if (mode == DMM_PR_FP32_KAHAN && block && ctx->bp_ready) return pr_bsum_blocks(ctx) + pr_bsplit_blocks(ctx);
  if (mode == DMM_PR_FP32_KAHAN && !block && ctx->tiles_ready) return pr_row_blocks(ctx);
  return pr_fused_blocks(ctx) + pr_super_blocks(ctx);
}

// One iteration on ctx->stream; the last one also reduces its own error.
// With gcontrib (a PE block's iteration from
// the global contribution vector) the FP32 modes may write the scores and
// the block's new contributions to score_out / contrib_out instead of the
// context's own buffers.
void launch_iteration(dmm_ctx* ctx, PrArgs a, int mode, int it, bool last, const void* gcontrib,
                      float* score_out = nullptr, float* contrib_out = nullptr, const PrHead* head = nullptr) {
  hipStream_t s = ctx->stream;
  const bool block_path = mode == DMM_PR_FP32_KAHAN && ctx->bp_ready && gcontrib;
  if (head && !block_path) hipLaunchKernelGGL(k_head, dim3(1), dim3(64), 0, s, *head);
  const int sb = a.super_blocks;
  // The error partials alternate between two halves: a kernel that writes its
  // own may still be reading the previous iteration's.
  double* const part0 = a.err_part;
  PrPrev prev{part0 + (it & 1 ? 0 : ctx->err_part_half), 0, it, a.ctrl, a.err_trace, a.prm};
  if (it & 1) a.err_part = part0 + ctx->err_part_half;
  prev.parts = pr_error_parts(ctx, mode, gcontrib != nullptr);
  float* const score_f = score_out ? score_out : ctx->d_score;
  if (mode == DMM_PR_FP32_SERIAL) {
    const float* cin = gcontrib ? static_cast<const float*>(gcontrib) : ctx->d_contrib[it & 1];
    float* cout = contrib_out ? contrib_out : ctx->d_contrib[(it + 1) & 1];
    a.main_blocks = pr_serial_blocks(ctx);
    a.super_blocks = 0;
    hipLaunchKernelGGL(k_serial, dim3(a.main_blocks), dim3(kSerialThreads), 0, s, a, prev, cin, cout, score_f);
  } else {
    const int fb = pr_fused_blocks(ctx);
    a.main_blocks = fb;
    if (mode == DMM_PR_FP64) {
      const double* cin = gcontrib ? static_cast<const double*>(gcontrib) : ctx->d_contrib64[it & 1];
      double* cout = ctx->d_contrib64[(it + 1) & 1];
      hipLaunchKernelGGL(k_fused<double>, dim3(fb), dim3(kFusedThreads), 0, s, a, prev, cin, cout, ctx->d_score64);
      hipLaunchKernelGGL(k_f64_super, dim3(sb), dim3(kThreads), 0, s, a, cout, ctx->d_score64);
    } else if (block_path) {
      const float* cin = static_cast<const float*>(gcontrib);
      float* cout = contrib_out ? contrib_out : ctx->d_contrib[(it + 1) & 1];
      BpArgs b;
      b.src = static_cast<const uint16_t*>(ctx->d_bp_src);
      b.wstart = static_cast<const int64_t*>(ctx->d_bp_wstart);
      b.wlen = static_cast<const int32_t*>(ctx->d_bp_wlen);
      b.wseg = static_cast<const int64_t*>(ctx->d_bp_wseg);
      b.wgroup = static_cast<const int64_t*>(ctx->d_bp_wgroup);
      b.groups = static_cast<const BlockGroup*>(ctx->d_bp_groups);
      b.seg_d = static_cast<const int32_t*>(ctx->d_bp_seg_d);
      b.brow = static_cast<const uint16_t*>(ctx->d_bp_brow);
      b.rows = static_cast<const FineRow*>(ctx->d_bp_rows);
      b.units = static_cast<const BlockUnit*>(ctx->d_bp_units);
      b.splits = static_cast<const BlockSplit*>(ctx->d_bp_splits);
      b.val = static_cast<float*>(ctx->d_bp_val);
      b.spare = b.val + ctx->m_in;
      b.part = static_cast<long long*>(ctx->d_bp_part);
      b.nwin = static_cast<int32_t>(ctx->n_bp_windows);
      // A block with fewer windows than CUs has several workgroups copy each.
      b.wparts = std::max<int32_t>(1, std::max(1, ctx->cu_count) / std::max(1, b.nwin));
      b.n_units = ctx->n_bp_units;
      b.n_splits = ctx->n_bp_splits;
      hipLaunchKernelGGL(k_bprop, dim3(std::max(1, ctx->cu_count)), dim3(kBPropThreads), 0, s, b, cin, a.n_gather,
                         head ? *head : PrHead{});
      a.main_blocks = pr_bsum_blocks(ctx);
      a.super_blocks = pr_bsplit_blocks(ctx);
      if (ctx->bp_fine)
        hipLaunchKernelGGL(k_bfine, dim3(a.main_blocks), dim3(kBSumThreads), 0, s, a, b, cout, score_f);
      else
        hipLaunchKernelGGL(k_bsum, dim3(a.main_blocks), dim3(kBSumThreads), 0, s, a, b, cout, score_f);
      if (a.super_blocks > 0)
        hipLaunchKernelGGL(k_bsplit, dim3(a.super_blocks), dim3(kThreads), 0, s, a, b, cout, score_f);
    } else if (ctx->tiles_ready && !gcontrib) {
      const float* cin = ctx->d_contrib[it & 1];
      float* cout = ctx->d_contrib[(it + 1) & 1];
      TileArgs t;
      t.cwin = ctx->d_wt_cwin;
      t.wstart = ctx->d_wt_wstart;
      t.cbase = ctx->d_wt_cbase;
      t.meta = ctx->d_wt_meta;
      t.src = ctx->d_wt_src;
      t.n_chunks = ctx->n_chunks;
      t.part = static_cast<float*>(ctx->d_wt_part);
      t.brow = ctx->d_wt_brow;
      t.bseg = ctx->d_wt_bseg;
      t.bsize = ctx->d_wt_bsize;
      t.seg_start = ctx->d_wt_seg_start;
      t.seg_off = ctx->d_wt_seg_off;
      t.istart = ctx->d_wt_istart;
      t.idx = ctx->d_wt_idx;
      t.n_blocks = ctx->n_row_blocks;
      const int tb = std::max(1, ctx->cu_count);
      if (ctx->tiles_window == 16384)
        hipLaunchKernelGGL(k_tile<16384>, dim3(tb), dim3(kTileThreads), 0, s, t, prev, cin, a.n_gather);
      else
        hipLaunchKernelGGL(k_tile<32768>, dim3(tb), dim3(kTileThreads), 0, s, t, prev, cin, a.n_gather);
      a.main_blocks = pr_row_blocks(ctx);
      a.super_blocks = 0;
      hipLaunchKernelGGL(k_rows, dim3(a.main_blocks), dim3(kRowThreads), 0, s, a, t, cout, ctx->d_score);
    } else {
      const float* cin = gcontrib ? static_cast<const float*>(gcontrib) : ctx->d_contrib[it & 1];
      float* cout = contrib_out ? contrib_out : ctx->d_contrib[(it + 1) & 1];
      hipLaunchKernelGGL(k_fused<float>, dim3(fb), dim3(kFusedThreads), 0, s, a, prev, cin, cout, score_f);
      hipLaunchKernelGGL(k_kahan_super, dim3(sb), dim3(kThreads), 0, s, a, cout, score_f);
    }
  }
  // A block's one iteration with a single k_bsplit workgroup is reduced by that.
  if (last && !(block_path && a.super_blocks == 1)) hipLaunchKernelGGL(k_reduce, dim3(1), dim3(kThreads), 0, s, a);
}

}  // namespace

int pr_light_blocks(dmm_ctx* ctx) {
  return static_cast<int>(std::max<int64_t>(
      1, std::min<int64_t>(int64_t(std::max(1, ctx->cu_count)) * 8, ceil_div(ctx->nloc, kThreads))));
}

// Deals the rows to the serial kernel's workgroups: longest first, each to
// the workgroup with the fewest edges so far (the first of equals).  Static, so
// that every run adds the error terms in the same order.  heavy: the heavy
// rows in order; by_class: longest power-of-two class first.  Part of every
// upload, so a deal is one sift of a heap's top (131 K vertices, 2048 bundles:
// 70 us; 250 with a pop and a push each and every row's length looked at).
void serial_plan(int64_t rows, int64_t light_begin, int64_t zero_begin, const int64_t* off,
                 const std::vector<int32_t>& heavy, const std::vector<int32_t>& by_class, int blocks,
                 std::vector<SerialItem>* items, std::vector<int32_t>* start) {
  struct Load {
    int64_t edges;
    int32_t block;
    bool operator<(const Load& o) const { return edges != o.edges ? edges < o.edges : block < o.block; }
  };
  std::vector<Load> heap(blocks);  // the least at the top
  for (int32_t b = 0; b < blocks; b++) heap[b] = {0, b};
  struct Dealt {
    SerialItem it;
    int32_t block;
  };
  std::vector<Dealt> dealt;
  dealt.reserve(by_class.size() + static_cast<size_t>(ceil_div(zero_begin - light_begin, kLightBundle)));
  auto deal = [&](int32_t first, int32_t kind, int64_t edges) {
    Load top = heap[0];
    dealt.push_back({{first, kind}, top.block});
    top.edges += edges;
    size_t at = 0;
    for (size_t kid; (kid = 2 * at + 1) < heap.size(); at = kid) {
      if (kid + 1 < heap.size() && heap[kid + 1] < heap[kid]) kid++;
      if (top < heap[kid]) break;
      heap[at] = heap[kid];
    }
    heap[at] = top;
  };
  auto len = [&](int64_t r) { return off[r + 1] - off[r]; };
  const int64_t off_end = off[rows];
  constexpr int64_t kItemCost = 128;  // an item's own steps, in edges
  int64_t block_row = kSerialBlockRow;
  while (block_row > kSerialBlockLeast && block_row * blocks > off_end) block_row /= 2;
  size_t h = 0;
  for (; h < by_class.size() && len(by_class[h]) >= block_row; h++)
    deal(by_class[h], kSerialBlock, len(by_class[h]));
  for (; h < by_class.size() && len(by_class[h]) >= kSerialWaveRow; h++)
    deal(by_class[h], kSerialWave, len(by_class[h]) + kItemCost);
  for (; h < by_class.size(); h += kHeavyBundle) {
    int64_t edges = 0;
    for (size_t i = h; i < std::min(by_class.size(), h + kHeavyBundle); i++) edges += len(by_class[i]);
    deal(static_cast<int32_t>(h), kSerialHeavy, edges + kItemCost);
  }
  size_t k = 0;
  while (k < heavy.size() && heavy[k] < light_begin) k++;
  for (int64_t r = light_begin; r < zero_begin; r += kLightBundle) {
    const int64_t end = std::min(zero_begin, r + kLightBundle);
    int64_t edges = off[end] - off[r];
    for (; k < heavy.size() && heavy[k] < end; k++) edges -= len(heavy[k]);
    deal(static_cast<int32_t>(r), kSerialLight, edges + kItemCost);
  }
  start->assign(blocks + 1, 0);
  for (const Dealt& d : dealt) (*start)[d.block + 1]++;
  for (int b = 0; b < blocks; b++) (*start)[b + 1] += (*start)[b];
  items->resize(dealt.size());
  std::vector<int32_t> at(start->begin(), start->end() - 1);
  for (const Dealt& d : dealt) (*items)[at[d.block]++] = d.it;
}

int pr_serial_blocks(dmm_ctx* ctx) { return std::max(1, ctx->cu_count); }

int pr_fused_blocks(dmm_ctx* ctx) {
  const int64_t lanes = std::max(ctx->nloc * kGroup, ctx->n_items * 64);
  return static_cast<int>(
      std::max<int64_t>(1, std::min<int64_t>(std::max(1, ctx->cu_count), ceil_div(lanes, kFusedThreads))));
}

int pr_row_blocks(dmm_ctx* ctx) { return kRowGroupsPerCU * std::max(1, ctx->cu_count); }

int pr_bsum_blocks(dmm_ctx* ctx) {
  const int64_t per_cu = ctx->bp_fine ? 2 : 1;  // by LDS
  return static_cast<int>(
      std::max<int64_t>(1, std::min<int64_t>(per_cu * std::max(1, ctx->cu_count), ctx->n_bp_units)));
}

int pr_bsplit_blocks(dmm_ctx* ctx) { return static_cast<int>(ceil_div(ctx->n_bp_splits, kThreads)); }

int pr_super_blocks(dmm_ctx* ctx) {
  return static_cast<int>(std::max<int64_t>(1, ceil_div(ctx->n_super, kThreads)));
}

int pr_run(dmm_ctx* ctx, int32_t max_iters, double epsilon, int32_t mode, dmm_pr_stats* stats) {
  // Constants exactly as the reference computes them in float
  // (src/pr.cc:39, 45-46), widened for the FP64 mode.
  PrParams* p = reinterpret_cast<PrParams*>(ctx->h_prparams);
  const float kDamp = 0.85f;
  const float nf = static_cast<float>(ctx->n);
  p->eps = epsilon;
  p->damp_f = kDamp;
  p->base_f = (1.0f - kDamp) / nf;
  p->init_f = 1.0f / nf;
  p->damp_d = static_cast<double>(kDamp);
  p->base_d = static_cast<double>(p->base_f);
  p->init_d = static_cast<double>(p->init_f);
  p->pad = 0;
  DMM_HIP_CHECK(ctx, hipMemcpyAsync(ctx->d_prparams, ctx->h_prparams, sizeof(PrParams),
                                    hipMemcpyHostToDevice, ctx->stream));
  // Two captured graphs per (mode, max_iters): init and the iterations that
  // the last runs took (at first max_iters), and what is left up to max_iters,
  // captured and launched once a run does not converge within the first.
  // Iterations after convergence return at once, but their launches take 5 us
  // a kernel: 16 K Kronecker vertices, 9 iterations of at most 20: 279 -> 251
  // us a call.
  const int key = mode * 100000 + max_iters;
  if (ctx->pr_graph_key != key) ctx->pr_runs = ChainRuns();
  const int most = ctx->pr_runs.most();
  const int want = most > 0 ? std::min(most, max_iters) : max_iters;
  const PrArgs a = make_args(ctx);
  auto capture = [&](hipGraphExec_t* exec, int first, int end) {
    return capture_chain(ctx, "PR", exec, [&] {
      const int ib = pr_light_blocks(ctx);
      if (first == 0) {
        if (mode == DMM_PR_FP64)
          hipLaunchKernelGGL(k_init_f64, dim3(ib), dim3(kThreads), 0, ctx->stream, a, ctx->d_score64,
                             ctx->d_contrib64[0]);
        else
          hipLaunchKernelGGL(k_init_f32, dim3(ib), dim3(kThreads), 0, ctx->stream, a, ctx->d_score,
                             ctx->d_contrib[0]);
      }
      for (int it = first; it < end; it++) launch_iteration(ctx, a, mode, it, it + 1 == end, nullptr);
      // Scores back to the caller's IDs.
      if (ctx->relabeled) {
        if (mode == DMM_PR_FP64)
          launch_map_scores_f64(ctx);
        else
          launch_map_scores_f32(ctx);
      }
    });
  };
  OldGraphs old;
  if (!ctx->pr_graph || ctx->pr_graph_key != key || ctx->pr_runs.anew(want, ctx->pr_chain)) {
    old.take(ctx->pr_graph, ctx->pr_rest);
    int rc = capture(&ctx->pr_graph, 0, want);
    if (rc) return rc;
    ctx->pr_graph_key = key;
    ctx->pr_chain = want;
    ctx->pr_runs.lost = 0;
  }
  double* h_trace = reinterpret_cast<double*>(ctx->h_prctrl + 1);
  const int trace = std::min(max_iters, DMM_MAX_PR_ITERS);
  DMM_HIP_CHECK(ctx, hipEventRecord(ctx->ev_a, ctx->stream));
  int waits = 0;
  for (int part = 0; part < 2; part++) {
    if (part == 1 && !ctx->pr_rest) {
      int rc = capture(&ctx->pr_rest, ctx->pr_chain, max_iters);
      if (rc) return rc;
    }
    DMM_HIP_CHECK(ctx, hipGraphLaunch(part == 0 ? ctx->pr_graph : ctx->pr_rest, ctx->stream));
    old.drop();
    DMM_HIP_CHECK(ctx, hipEventRecord(ctx->ev_b, ctx->stream));
    DMM_HIP_CHECK(ctx, hipMemcpyAsync(ctx->h_prctrl, ctx->d_prctrl, sizeof(PrCtrl), hipMemcpyDeviceToHost,
                                      ctx->stream));
    // The error trace too: one wait for both.
    if (stats && trace > 0)
      DMM_HIP_CHECK(ctx, hipMemcpyAsync(h_trace, ctx->d_err_trace, sizeof(double) * trace, hipMemcpyDeviceToHost,
                                        ctx->stream));
    DMM_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    waits = part;
    if (ctx->pr_chain == max_iters || ctx->h_prctrl->pad) break;
  }
  ctx->pr_runs.add(static_cast<int>(ctx->h_prctrl->ticket), ctx->pr_chain, mode == DMM_PR_FP32_SERIAL ? 1 : 2, waits);
  ctx->pr_mode = mode;
  if (stats) {
    float ms = 0;
    DMM_HIP_CHECK(ctx, hipEventElapsedTime(&ms, ctx->ev_a, ctx->ev_b));
    const int iters = static_cast<int>(ctx->h_prctrl->ticket);
    stats->iters = iters;
    stats->total_ms = ms;
    stats->iter_ms = iters > 0 ? ms / iters : 0;
    std::copy(h_trace, h_trace + std::min(iters, trace), stats->err);
    const int64_t m = ctx->m_in, nl = ctx->nloc;
    stats->alg_bytes_per_iter = (mode == DMM_PR_FP64) ? 12 * m + 32 * nl + 8 : 8 * m + 20 * nl + 8;
  }
  return DMM_OK;
}

int pr_block_iteration(dmm_ctx* ctx, const float* gcontrib_host, float* scores_inout, int32_t mode,
                       double* err, double* ms) {
  if (!ctx->d_gcontrib) {
    int rc = dev_alloc(ctx, reinterpret_cast<void**>(&ctx->d_gcontrib), sizeof(float) * ctx->n,
                       "global contribution vector");
    if (rc) return rc;
  }
  PrParams* p = reinterpret_cast<PrParams*>(ctx->h_prparams);
  const float kDamp = 0.85f;
  const float nf = static_cast<float>(ctx->n);
  p->eps = -1.0;
  p->damp_f = kDamp;
  p->base_f = (1.0f - kDamp) / nf;
  p->init_f = 1.0f / nf;
  p->damp_d = static_cast<double>(kDamp);
  p->base_d = static_cast<double>(p->base_f);
  p->init_d = static_cast<double>(p->init_f);
  DMM_HIP_CHECK(ctx, hipMemcpyAsync(ctx->d_prparams, ctx->h_prparams, sizeof(PrParams),
                                    hipMemcpyHostToDevice, ctx->stream));
  DMM_HIP_CHECK(ctx, hipMemcpyAsync(ctx->d_gcontrib, gcontrib_host, sizeof(float) * ctx->n,
                                    hipMemcpyHostToDevice, ctx->stream));
  DMM_HIP_CHECK(ctx, hipMemcpyAsync(ctx->d_score, scores_inout, sizeof(float) * ctx->nloc,
                                    hipMemcpyHostToDevice, ctx->stream));
  hipLaunchKernelGGL(k_reset_ctrl, dim3(1), dim3(1), 0, ctx->stream, ctx->d_prctrl);
  PrArgs a = make_args(ctx);
  // The timed region starts after the host copies have landed.
  DMM_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  DMM_HIP_CHECK(ctx, hipEventRecord(ctx->ev_a, ctx->stream));
  launch_iteration(ctx, a, mode, 0, true, ctx->d_gcontrib);
  DMM_HIP_CHECK(ctx, hipEventRecord(ctx->ev_b, ctx->stream));
  DMM_HIP_CHECK(ctx, hipGetLastError());
  DMM_HIP_CHECK(ctx, hipMemcpyAsync(scores_inout, ctx->d_score, sizeof(float) * ctx->nloc,
                                    hipMemcpyDeviceToHost, ctx->stream));
  DMM_HIP_CHECK(ctx, hipMemcpyAsync(ctx->h_prctrl, ctx->d_prctrl, sizeof(PrCtrl), hipMemcpyDeviceToHost,
                                    ctx->stream));
  DMM_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  if (err) *err = ctx->h_prctrl->err;
  if (ms) {
    float f = 0;
    DMM_HIP_CHECK(ctx, hipEventElapsedTime(&f, ctx->ev_a, ctx->ev_b));
    *ms = f;
  }
  return DMM_OK;
}

// ---- allocation-free PE-block iteration -------------------------------------
//
// The same kernels as pr_block_iteration, with everything they need beyond
// the caller's buffers and the uploaded graph -- constants, control block,
// error partials, split-row segment partials -- in one file-scope device
// array.  Each GPU holds its own copy of the array for the life of the
// process; host code reaches it only through the address hipGetSymbolAddress
// returns for that device (scratch_ptr), never through the array's name.
// Calls that overlap on one GPU share it and race.

namespace {

constexpr size_t kScratchBytes = size_t(4) << 20;  // per GPU
constexpr size_t kScratchParams = 0;                // PrParams
constexpr size_t kScratchCtrl = 64;                 // PrCtrl
constexpr size_t kScratchTrace = 96;                // one error-trace entry
constexpr size_t kScratchErr = 256;                 // error partials
constexpr int kScratchErrParts = 8192;
constexpr size_t kScratchSegs = kScratchErr + sizeof(double) * kScratchErrParts;  // segment partials
constexpr int64_t kScratchSegCap = static_cast<int64_t>((kScratchBytes - kScratchSegs) / sizeof(double2));
static_assert(sizeof(PrParams) <= kScratchCtrl && sizeof(PrCtrl) <= kScratchTrace - kScratchCtrl, "scratch head");

}  // namespace

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {

constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
unsigned char* g_scratch_ptr[kMaxScratchDevices] = {};

}  // namespace

int scratch_init(dmm_ctx* ctx) {
  if (ctx->device < 0 || ctx->device >= kMaxScratchDevices)
    return set_err(ctx, DMM_ERR_INVALID, "device %d beyond the scratch table", ctx->device);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[ctx->device]) {
    void* p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return set_err(ctx, DMM_ERR_HIP, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
    g_scratch_ptr[ctx->device] = static_cast<unsigned char*>(p);
  }
  ctx->scratch = g_scratch_ptr[ctx->device];
  return DMM_OK;
}

int pr_block_iteration_noalloc(dmm_ctx* ctx, const float* d_gcontrib, float* d_scores, float* d_contrib_out,
                               int32_t mode, double* d_err) {
  unsigned char* base = ctx->scratch;
  if (!base) return set_err(ctx, DMM_ERR_STATE, "the context has no scratch address");
  PrArgs a = make_args(ctx);
  const int parts = pr_error_parts(ctx, mode, true);
  if (parts > kScratchErrParts)
    return set_err(ctx, DMM_ERR_CAPACITY, "%d error partials exceed the %d the scratch array holds", parts,
                   kScratchErrParts);
  if (ctx->n_slots > kScratchSegCap)
    return set_err(ctx, DMM_ERR_CAPACITY, "%lld split-row segments exceed the %lld the scratch array holds",
                   (long long)ctx->n_slots, (long long)kScratchSegCap);
  a.prm = reinterpret_cast<const PrParams*>(base + kScratchParams);
  a.ctrl = reinterpret_cast<PrCtrl*>(base + kScratchCtrl);
  a.err_trace = reinterpret_cast<double*>(base + kScratchTrace);
  a.err_out = d_err;
  a.err_part = reinterpret_cast<double*>(base + kScratchErr);
  a.partial = reinterpret_cast<double2*>(base + kScratchSegs);
  // Constants as the reference computes them in float (src/pr.cc:39, 45-46);
  // no convergence test (one iteration).
  PrHead head;
  head.prm = reinterpret_cast<PrParams*>(base + kScratchParams);
  head.ctrl = a.ctrl;
  PrParams& p = head.p;
  const float kDamp = 0.85f;
  const float nf = static_cast<float>(ctx->n);
  p.eps = -1.0;
  p.damp_f = kDamp;
  p.base_f = (1.0f - kDamp) / nf;
  p.init_f = 1.0f / nf;
  p.damp_d = static_cast<double>(kDamp);
  p.base_d = static_cast<double>(p.base_f);
  p.init_d = static_cast<double>(p.init_f);
  p.pad = 0;
  launch_iteration(ctx, a, mode, 0, true, d_gcontrib, d_scores, d_contrib_out, &head);
  DMM_HIP_CHECK(ctx, hipGetLastError());
  DMM_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  return DMM_OK;
}

}  // namespace dmm
