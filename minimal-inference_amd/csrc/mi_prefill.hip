// Ragged (varlen) causal prefill attention over the paged pool, bf16 MFMA.
//
// Reference: the prefill wrapper's plan() (scheduler.py:704-716: qo_indptr,
// paged_kv_indptr / indices / last_page_len, causal=True) and run()
// (model.py:235, mode == "prefill").  Query row i of request b sees KV tokens
// j <= i + (kv_len - qo_len); the reference always has kv_len == qo_len.
//
// Work decomposition.  A workgroup (4 waves) owns `bm` query positions of one
// request and ALL `group` Q heads of one KV head: bm x group (position, head)
// rows in position-major order, cut into row blocks of 16 rows dealt to the
// waves round robin (three per wave for head_dim 128, two for 64, one for 256,
// computed together so every K / V operand read from LDS feeds all of them).
// bm = rows / group (192 rows for head_dim 128: 24 positions for group 8, 48
// for group 4), so every K/V byte the workgroup stages serves all the heads
// of its group.  (8-wave workgroups over twice the positions halve the
// staging per wave but measured 10 % slower: two independent 4-wave
// workgroups per CU keep computing across each other's barriers.)  Launches
// that leave most of the chip idle take fine tiles of one row block per wave
// instead, and tiles with long key ranges are cut into units along the keys
// whose fp32 partials the last unit merges (prefill_plan_kernel says when and
// why).  plan() lists the tiles, and where it pays the units, request
// by request (longest prompt first), each request's tiles heaviest first; the
// grid maps them tile-major, so the XCD that a KV head's workgroups land on runs
// one request's tiles back to back and finds its K / V in L2.  The units'
// partials lie in the workspace, so only runs in the order of the plan's stream
// use them; every other run takes the tiles and only reads the workspace
// (RunKey).
//
// Per 64-key tile: the workgroup stages K and V in LDS (double buffered: the
// next tile's global loads are in flight while this one is consumed; one
// barrier per tile); each wave, per row block:
//   S^T = K Q^T  -- 16x16x32 MFMAs, K rows read from LDS as the A operand,
//                   Q^T held in registers as B; lane (g, n) gets
//                   S^T[key 4g+i][row n] for each 16-key block;
//   online softmax per row in the exp2 domain with a lazy running max
//   (rescale only when the max grows by more than 2^8); row maxima across
//   lane groups with the gfx950 lane-swap instructions;
//   O += P V     -- 16x16x32 MFMAs over 32 keys: the S^T accumulators of two
//                   key blocks are exactly the P operand (lane (g, n) holds
//                   keys {4g+i} of both), and V comes from the gfx950 LDS
//                   transpose read in the same key order.
#include <math.h>

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "mi_common.h"

namespace {

// s_waitcnt immediate (gfx9 encoding): vmcnt = 0, expcnt = 7, lgkmcnt = 15.
constexpr int kWaitVmcnt0 = 0x0F70;
// Buffer resource word 3 for gfx9 raw buffers (32-bit data format, no swizzle).
constexpr int kBufferWord3 = 0x00020000;

constexpr int kPageSize = 16;
constexpr int kMinRows = 8;    // fewest query positions per workgroup (head_dim 256, group 8)
constexpr int kKvTile = 64;    // keys per staged tile (4 pages)
constexpr float kLazyRescale = 8.0f;
// K / V tiles staged straight to LDS by the gfx950 buffer loads with the
// `lds` modifier (no staging registers, no LDS store instructions).  A wave's
// load instruction fills 1 KB of LDS, lane l at byte 16 l, so the rows are
// unpadded and a 16-byte chunk's place in its row is permuted instead
// (chunk_slot) to keep the reads off shared banks.
// Output staging: pad bytes after every 8 columns (32 bytes each) of a
// column-major 16-row block, so the 8-byte writes of a half wave and the
// transpose reads of two lane groups fall on distinct banks.
constexpr int kOutPad = 144;

// One work unit of the run: the KV tiles [kt_begin, kt_end) of one query tile.
// A query tile whose keys are cut into `nsplit` > 1 units has consecutive
// units, each with its own partial slot.
struct alignas(32) PrefillTile {
  int q_begin;  // absolute first query row of the tile
  int q_rows;   // positions in this tile (<= bm)
  int qo_len;
  int kv_len;
  int row0;           // first position of the tile within its request
  int kv_page_begin;  // absolute position of the request's first page in kv_indices
  int kt;             // kt_begin | kt_end << 16 (kToEnd: to the tile's last key)
  int part;           // partial slot << 16 | split << 8 | nsplit (nsplit <= 1: the whole tile)
};
constexpr unsigned kToEnd = 0xffffu;

// Which runs may take the units of a plan: the partials and their counters
// belong to one run at a time, and nothing but the order of a stream says that
// two runs do not overlap.  So a run takes the units only on the stream the plan
// was made on, with the plan's workspace (address and size: a copy of a
// workspace has no partials of its own) and geometry, and outside of graph
// capture (a graph's replays are ordered with nothing else); the plan's
// `serial`, in the header and in front of the units, tells a header that was put
// back over a later plan's units.  Every other run takes the tile list, which
// needs the workspace's first mi_prefill_workspace_size bytes only and writes
// none of them.
struct RunKey {
  uint64_t ws, bytes, stream, shape;
};

struct PrefillHeader {
  int num_tiles;   // whole coarse tiles, behind the header
  int error;
  int bm;          // query positions per tile of the units
  int row_blocks;  // their 16-row blocks per wave: the coarse or the fine form
  int chunk;       // KV tiles per unit at most (0: no tile is split)
  int slots;       // partial slots per KV head (the counters follow them)
  int units;       // 0: every run takes the tiles
  int pad;
  RunKey key;
  uint64_t serial;
};
static_assert(sizeof(PrefillHeader) <= 256, "the tiles start at byte 256");

// Waves per workgroup.
constexpr int waves_for(int /*head_dim*/) { return 4; }

// Row blocks of 16 (position, head) rows per wave of the coarse tiles: three
// for head_dim 128 (each K / V operand read from LDS then feeds three blocks),
// two for 64, one for 256.  The fine tiles have one.
constexpr int row_blocks(int head_dim) { return head_dim > 128 ? 1 : head_dim == 128 ? 3 : 2; }

// Query positions per workgroup: the workgroup's 16 * waves * row blocks rows
// hold bm positions x group heads, bm = rows / group.
int rows_per_tile(int group, int head_dim, int blocks) { return 16 * waves_for(head_dim) * blocks / group; }

size_t tile_capacity(int batch, int64_t total_q) { return size_t(total_q / kMinRows + batch + 1); }

size_t prefill_ws_bytes(int batch, int64_t total_q) {
  return 256 + mi::align_up(tile_capacity(batch, total_q) * sizeof(PrefillTile), 256);
}

// Workgroups resident at once, as the plan counts them: two per CU at head_dim 128
// (registers), one at 256 (LDS), three of the four that fit at 64 (filling the
// fourth place with splits, one prompt of 1,537 tokens, Qwen2.5-0.5B heads, took
// 19.6 us instead of 15.7).
int resident_groups(int cus, int head_dim) { return cus * (head_dim == 64 ? 3 : head_dim == 128 ? 2 : 1); }

// Fine tiles are for launches that leave most of the chip idle: a KV tile
// takes a workgroup of one row block per wave 1.1-1.3 us instead of the 2.2-2.8
// us of three, so a chain of them is half as long and a merge moves a third of
// the bytes, but the K / V operands read from LDS feed a third of the MFMAs.
// Measured on Mistral-7B heads, whole coarse tiles / coarse and split / fine
// (and split): one prompt of 512 tokens 23.9 / 21.8 / 13.5 us, 1,024: 41.0 /
// 36.2 / 25.3, 64 new tokens on 8,000 cached 267 / 66.5 / 31.7; 2,048: 79 / 54 /
// 60; four turns of 61-413 tokens on 2,000-6,000 cached 199 / 89 / 132;
// Qwen2.5-7B heads, one prompt of 1,537: 59 / 41 / 44.  So: fine while the load per
// resident workgroup, counted in fine KV tiles, is at most kFineLoad.
//
// Fine tiles of more than one resident round must pay for the rounds as well: they
// are taken only where rows and longest chain make them no slower than coarse
// tiles at the same cost per KV tile, load + longest / 2 <= max(longest, load +
// longest / 2) with the loads in each form's own tiles (a chain is on average
// half the longest when it starts).  Of 500 launches of 1-64 requests with up to
// four rounds of fine tiles, 18 of head_dim 128 were up to 20 % slower in fine
// tiles than in the whole coarse ones (32 requests of 20 rows on 500 cached,
// Qwen2.5-72B heads, 27.3 / 32.2 us; 32 of 300 on 100, 8 KV heads of one, 31.6 /
// 34.3), with this line three, by at most 7 %.  Coarse tiles of a launch below the load line are
// not split: at few KV tiles per workgroup the partials of three row blocks cost
// more than the chain (five prompts of 307, Qwen2.5-7B heads, 17.5 whole, 25.3 split).
constexpr int kFineLoad = 12;
constexpr int kFineRounds = 4;  // resident rounds of fine units at most

// Workgroups of the run: whole resident rounds over the most coarse tiles the
// rows can make, or the units that a plan of fine tiles may hold.  The plan
// never makes more.
int64_t run_groups(int64_t res, int batch, int64_t total_q, int group, int hkv, int head_dim) {
  const auto groups = [&](int blocks) { return (total_q / rows_per_tile(group, head_dim, blocks) + batch) * hkv; };
  const int64_t coarse = (groups(row_blocks(head_dim)) + res - 1) / res * res;
  const int64_t fine = (groups(1) + res - 1) / res * res;
  return std::max(coarse, std::min(fine, kFineRounds * res));
}

// A split unit's partial, per KV head: the workgroup's O accumulators in lane
// order and (m, l) per lane and row block, all fp32.
constexpr size_t partial_bytes(int head_dim, int blocks) {
  return size_t(waves_for(head_dim)) * blocks * (head_dim / 16 * 1024 + 512);
}
constexpr int kCounterStride = 32;  // ints: one 128-byte line per merge counter
constexpr int kMaxSplits = 64;      // per tile

// The units and their partials: the end of the workspace, at most three
// quarters of it and two resident rounds of coarse units.  At `off` the serial
// of the plan whose units these are, 256 bytes further the units (room for
// kFineRounds resident rounds), at `parts` the partial slots (per KV head
// `coarse` of coarse or `fine` of fine units) and behind them the counters.  No
// slots when the workspace is too small to be worth it: the plan then makes
// tiles only.
struct UnitLayout {
  size_t off, parts;
  int capacity, coarse, fine;
};
UnitLayout unit_layout(int res, size_t workspace_bytes, int hkv, int head_dim) {
  const auto per = [&](int blocks) { return (partial_bytes(head_dim, blocks) + kCounterStride * sizeof(int)) * size_t(hkv); };
  UnitLayout L{0, 0, 0, 0, 0};
  const size_t coarse = per(row_blocks(head_dim)), limit = workspace_bytes / 4 * 3;
  const int capacity = kFineRounds * res / hkv;
  const size_t list = 256 + mi::align_up(size_t(capacity) * sizeof(PrefillTile), 256);
  const size_t c = limit < list ? 0 : std::min((limit - list) / coarse, size_t(2 * res / hkv));
  if (c < 2 || list + c * coarse + 512 + sizeof(PrefillTile) > workspace_bytes) return L;
  L.off = (workspace_bytes - c * coarse - list) & ~size_t(255);
  L.parts = L.off + list;
  L.capacity = capacity;
  L.coarse = int(c);
  L.fine = int(std::min(c * coarse / per(1), size_t(0xffff)));
  return L;
}

// The stream that orders the calls made on `s`, as RunKey has it: 0 for none
// (under capture the launch happens in replays on any stream; the per-thread
// default stream is one handle for many streams).
uint64_t ordering_stream(hipStream_t s) {
  if (s == hipStreamPerThread) return 0;
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &status) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return status == hipStreamCaptureStatusNone ? reinterpret_cast<uint64_t>(s) + 1 : 0;
}

RunKey run_key(const void* ws, size_t bytes, int hkv, int group, int head_dim, hipStream_t s) {
  return RunKey{reinterpret_cast<uint64_t>(ws), bytes, ordering_stream(s),
                uint64_t(unsigned(hkv)) << 32 | uint64_t(unsigned(group)) << 16 | uint64_t(unsigned(head_dim) & 0xffff)};
}

struct PlanParams {
  const int32_t* qo_indptr;
  const int32_t* kv_indptr;
  const int32_t* last_page_len;
  int batch;
  int capacity;
  int group, hkv;
  int bm[2], blocks[2], slots[2];  // positions, row blocks per wave and partial slots of fine [0] and coarse [1] tiles
  size_t counters_off[2];          // of the merge counters, behind the partials
  int resident;                    // workgroups resident at once
  int cus;                         // their number, where several workgroups share one (0: one each)
  int tile_room;                   // tiles the list holds in front of the units
  int unit_capacity;               // 0: tiles only
  char* ws;
  PrefillHeader* header;
  PrefillTile* tiles;
  PrefillTile* units;
  uint64_t* unit_serial;
  RunKey key;
  uint64_t serial;
};

constexpr int kPlanThreads = 1024;
constexpr int kSplitTiles = 8192;  // most query tiles whose keys are considered for splitting
constexpr int kMinChunk = 4;  // KV tiles per unit at least (2 and 3 measured the same on a 512-token prompt)
// KV tiles that splitting must take off the longest chain: the partials cost about
// as much as two, and more where the whole tiles had a CU each and the units share
// them.  (us, whole / split: 16 requests of 16 rows on 300 cached, head_dim 256, five
// KV tiles to four, 16.2 / 18.2; Mistral-7B heads 9.9 / 11.6; 20 of 10 on 400, seven
// to four, 12.9 / 15.5.  One row on 400 cached, seven to four, most of the chip idle,
// 11.9 / 11.0; 900 tokens, Qwen2.5-7B heads, 15 to 12, 400 tiles, 23.5 / 19.0.)
constexpr int kMinSaved = 2, kMinSavedCrowd = 5;

// Inclusive scan over the block: shuffles inside each wave, then the wave
// totals through LDS.  *total gets the block-wide sum.
__device__ int block_scan(int v, int* wsum, int* total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(v, o);
    if (lane >= o) v += y;
  }
  __syncthreads();  // the previous call's readers are done with wsum
  if (lane == 63) wsum[w] = v;
  __syncthreads();
  int pre = 0, tot = 0;
  for (int i = 0; i < kPlanThreads / 64; ++i) {
    const int s = wsum[i];
    pre += (i < w) ? s : 0;
    tot += s;
  }
  *total = tot;
  return v + pre;
}

__device__ __forceinline__ int request_kv(const PlanParams& p, int b) {
  const int np = max(0, p.kv_indptr[b + 1] - p.kv_indptr[b]);
  return np > 0 ? (np - 1) * kPageSize + min(max(p.last_page_len[b], 1), kPageSize) : 0;
}

__device__ __forceinline__ PrefillTile make_tile(int bm, int qo, int kv, int q0, int pb0, int nt, int k) {
  PrefillTile tile;
  tile.row0 = (nt - 1 - k) * bm;
  tile.q_begin = q0 + tile.row0;
  tile.q_rows = min(bm, qo - tile.row0);
  tile.qo_len = qo;
  tile.kv_len = kv;
  tile.kv_page_begin = pb0;
  tile.kt = int(kToEnd << 16);
  tile.part = 0;
  return tile;
}

// `ntiles` coarse tiles, `fit` of them listed
__device__ __forceinline__ void write_header(const PlanParams& p, int ntiles, int fit, int form, int units, int chunk) {
  p.header->num_tiles = fit;
  p.header->error = ntiles > p.capacity ? 1 : 0;
  p.header->bm = p.bm[form];
  p.header->row_blocks = p.blocks[form];
  p.header->chunk = chunk;
  p.header->slots = p.slots[form];
  p.header->units = units;
  p.header->key = p.key;
  p.header->serial = p.serial;
  if (units > 0) *p.unit_serial = p.serial;
}

// Batches of more requests than the block has threads: one request per thread
// and round, its place found by counting the requests ordered before it in
// global memory; tiles only.
__device__ void plan_large(const PlanParams& p, int* wsum, int* s_fit) {
  const int t = threadIdx.x, bm = p.bm[1];
  int total = 0;
  if (t == 0) *s_fit = 0;
  __syncthreads();
  for (int base = 0; base < p.batch; base += blockDim.x) {
    const int b = base + t;
    int nt = 0, start = 0;
    if (b < p.batch) {
      const int qo = max(0, p.qo_indptr[b + 1] - p.qo_indptr[b]);
      nt = (qo + bm - 1) / bm;
      for (int c = 0; c < p.batch; ++c) {
        const int qc = max(0, p.qo_indptr[c + 1] - p.qo_indptr[c]);
        if (qc > qo || (qc == qo && c < b)) start += (qc + bm - 1) / bm;
      }
      if (start + nt <= p.capacity) {
        for (int k = 0; k < nt; ++k)
          p.tiles[start + k] = make_tile(bm, qo, request_kv(p, b), p.qo_indptr[b], p.kv_indptr[b], nt, k);
        atomicMax(s_fit, start + nt);
      }
    }
    int chunk_total = 0;
    block_scan(nt, wsum, &chunk_total);
    total += chunk_total;
  }
  __syncthreads();
  if (t == 0) write_header(p, total, *s_fit, 1, 0, 0);  // (a record that nothing wrote is never run)
}

// Tile order: requests by decreasing prompt length (ties by index), each
// request's tiles from the end of its prompt (most keys) to the start.  The
// run kernel maps consecutive tiles of one (request, KV head) to consecutive
// workgroups of one XCD, so they share the request's K / V in that XCD's L2.
//
// Splitting.  A tile's keys are a serial chain of KV tiles that take about as
// long whether one or two workgroups share the CU, so a launch of few tiles
// (one prompt, a short turn on a long cached context) lasts as long as its
// longest tile while most of the chip idles.  Tiles of more than `chunk` KV
// tiles are therefore cut into near-equal units whose partial results the last
// unit to finish merges.  chunk is the smallest value of at least
//   * the load that fills every resident workgroup evenly (so launches of many
//     rounds, whose tiles balance by themselves, split nothing),
//   * kMinChunk, and sqrt(longest / 2): a further split costs its merger about
//     half a KV tile,
// whose units fit the rounds that the unsplit tiles need.  Coarse tiles split
// only to fill one round (split over a second one, a 4,096-token prompt went
// 160 -> 168 us: the partials of three row blocks are 104 KB per unit).  The
// count assumes a causal run; the last
// unit of a tile takes whatever keys remain, so a non-causal run of the same
// plan is complete too.  The whole coarse tiles are listed in any case, for the
// runs that may not take the units (RunKey).
__global__ __launch_bounds__(kPlanThreads) void prefill_plan_kernel(PlanParams p) {
  __shared__ int s_qo[kPlanThreads], s_kv[kPlanThreads], s_q0[kPlanThreads], s_pb0[kPlanThreads];
  __shared__ int s_req[kPlanThreads], s_end[kPlanThreads], wsum[kPlanThreads / 64];
  __shared__ int red[2][kPlanThreads / 64], ok[2][kPlanThreads / 64], s_fit;
  __shared__ float s_sums[4][kPlanThreads / 64];
  __shared__ unsigned short s_n[kSplitTiles];
  if (p.batch > kPlanThreads) {
    plan_large(p, wsum, &s_fit);
    return;
  }
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  constexpr int NW = kPlanThreads / 64;
  int qo = 0;
  // this request's (row, key) pairs with half a KV tile of masked ones per row, its
  // fine tiles, and the KV tiles of its fine and its coarse ones
  enum { kArea, kFineTiles, kFineKv, kCoarseKv, kSums };
  float sums[kSums] = {};
  int most_kv = 0;
  if (t < p.batch) {
    const int q0 = p.qo_indptr[t], q1 = p.qo_indptr[t + 1], pb0 = p.kv_indptr[t], pb1 = p.kv_indptr[t + 1];
    const int lpl = p.last_page_len[t];
    const int np = max(0, pb1 - pb0);
    const int kv = np > 0 ? (np - 1) * kPageSize + min(max(lpl, 1), kPageSize) : 0;
    qo = max(0, q1 - q0);
    s_qo[t] = qo;
    s_q0[t] = q0;
    s_pb0[t] = pb0;
    s_kv[t] = kv;
    const float keys = max(0.f, float(kv) - 0.5f * float(qo)) + 0.5f * kKvTile;  // of a row, on average
    sums[kArea] = float(qo) * keys;
    sums[kFineTiles] = float((qo + p.bm[0] - 1) / p.bm[0]);
    sums[kFineKv] = sums[kFineTiles] * keys * (1.f / kKvTile);
    sums[kCoarseKv] = float((qo + p.bm[1] - 1) / p.bm[1]) * keys * (1.f / kKvTile);
    most_kv = qo > 0 ? kv : 0;
  }
  const int request_waves = (p.batch + 63) / 64;  // (the others would only slow these down)
  if (w < request_waves) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
#pragma unroll
      for (int k = 0; k < kSums; ++k) sums[k] += __shfl_xor(sums[k], o);
      most_kv = max(most_kv, __shfl_xor(most_kv, o));
    }
    if (lane == 0) {
#pragma unroll
      for (int k = 0; k < kSums; ++k) s_sums[k][w] = sums[k];
      red[0][w] = most_kv;
    }
  }
  if (t == 0) s_fit = 0;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kSums; ++k) sums[k] = 0.f;
#pragma nounroll
  for (int i = 0; i < request_waves; ++i) {
#pragma unroll
    for (int k = 0; k < kSums; ++k) sums[k] += s_sums[k][i];
    most_kv = max(most_kv, red[0][i]);
  }
  int rank = 0;
  for (int c = 0; c < p.batch; ++c) {
    const int qc = s_qo[c];
    rank += (qc > qo || (qc == qo && c < t)) ? 1 : 0;
  }
  if (t < p.batch) {
    s_req[rank] = t;
  }
  __syncthreads();
  // tiles up to the end of each request, in rank order
  int bm = p.bm[1];
  auto scan_tiles = [&]() {
    int total = 0;
    const int end = block_scan(t < p.batch ? (s_qo[s_req[t]] + bm - 1) / bm : 0, wsum, &total);
    s_end[t] = end;
    if (t < p.batch && end <= p.capacity) atomicMax(&s_fit, end);
    __syncthreads();
    return total;
  };
  int ntiles = scan_tiles();
  const int coarse_tiles = ntiles, fit = s_fit;  // fit: tiles of the requests that fit the list

  // tile i of the list: its request's rank, and its causal KV tiles
  auto rank_of = [&](int i) {
    int lo = 0, hi = p.batch - 1;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (s_end[mid] > i) hi = mid; else lo = mid + 1;
    }
    return lo;
  };
  auto tile_of = [&](int i) {
    const int r = rank_of(i), b = s_req[r];
    const int nt = (s_qo[b] + bm - 1) / bm;
    return make_tile(bm, s_qo[b], s_kv[b], s_q0[b], s_pb0[b], nt, i - (s_end[r] - nt));
  };
  auto kv_tiles = [&](const PrefillTile& x) {
    return (max(0, min(x.kv_len, x.row0 + x.q_rows + x.kv_len - x.qo_len)) + kKvTile - 1) / kKvTile;
  };
  for (int i = t; i < fit; i += kPlanThreads) p.tiles[i] = tile_of(i);
  // fine or coarse units (see kFineLoad)
  const bool room = p.unit_capacity > 0 && ntiles == fit && fit <= p.tile_room;
  const float per_group = float(p.hkv) / float(p.resident), chain = float((most_kv + kKvTile - 1) / kKvTile);
  const bool light = sums[kArea] * float(p.group) * per_group <= 64.f * kKvTile * float(kFineLoad);
  const float rounds_fine = sums[kFineTiles] * per_group;
  const bool even = sums[kFineKv] * per_group + 0.5f * chain <= max(chain, sums[kCoarseKv] * per_group + 0.5f * chain);
  const int form =
      room && p.blocks[1] > 1 && light && rounds_fine <= float(kFineRounds) && (rounds_fine <= 1.f || even) ? 0 : 1;
  const int nslots = p.slots[form];
  if (form == 0) {
    __syncthreads();  // s_end's readers are done
    bm = p.bm[0];
    ntiles = scan_tiles();
  }
  // the units that fill the rounds which the unsplit tiles need
  const int rounds = (ntiles * p.hkv + p.resident - 1) / p.resident;
  const int limit = min(rounds * p.resident / p.hkv, p.unit_capacity);
  const bool consider = room && (form == 0 || (rounds == 1 && (!light || p.blocks[1] == 1))) && ntiles <= min(kSplitTiles, limit);
  int chunk = 0, longest = 0;
  if (consider) {
    int sum = 0;
    for (int i = t; i < ntiles; i += kPlanThreads) {
      const int n = kv_tiles(tile_of(i));
      s_n[i] = (unsigned short)min(n, 65535);
      sum += n;
      longest = max(longest, n);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      sum += __shfl_xor(sum, o);
      longest = max(longest, __shfl_xor(longest, o));
    }
    if (lane == 0) {
      red[0][w] = sum;
      red[1][w] = longest;
    }
    __syncthreads();
    long long total = 0;
    for (int i = 0; i < NW; ++i) {
      total += red[0][i];
      longest = max(longest, red[1][i]);
    }
    int lo = max(kMinChunk, int((total * p.hkv + p.resident - 1) / p.resident));
    lo = max(lo, max((longest + kMaxSplits - 1) / kMaxSplits, int(sqrtf(0.5f * float(longest)))));
    int hi = longest;
    if (longest < int(kToEnd)) {
      // every wave tries one value between lo and hi per round; the units and
      // the partial slots fall as the value grows, and `longest` fits
      for (int round = 0; lo < hi; ++round) {
        const int c = lo + (w + 1) * (hi - lo) / (NW + 1);
        int units = 0, parts = 0;
        for (int i = lane; i < ntiles; i += 64) {
          const int ns = max(1, (int(s_n[i]) + c - 1) / c);
          units += ns;
          parts += ns > 1 ? ns : 0;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
          units += __shfl_xor(units, o);
          parts += __shfl_xor(parts, o);
        }
        if (lane == 0) ok[round & 1][w] = units <= limit && parts <= nslots;
        __syncthreads();
        int nlo = lo, nhi = hi;
        for (int i = 0; i < NW; ++i) {
          const int ci = lo + (i + 1) * (hi - lo) / (NW + 1);
          if (ok[round & 1][i]) nhi = min(nhi, ci); else nlo = max(nlo, ci + 1);
        }
        lo = nlo;
        hi = nhi;
      }
      // (kMinSaved)
      const bool crowd = float(ntiles * p.hkv) <= float(p.cus) &&
                         (float(total) / float(lo) + 0.5f * float(ntiles)) * float(p.hkv) > float(p.cus);
      chunk = lo + (crowd ? kMinSavedCrowd : kMinSaved) <= longest ? lo : 0;
    }
  }
  // whole fine tiles are units, whole coarse ones the tiles that are listed already
  int units = form == 0 && ntiles <= p.unit_capacity ? ntiles : 0;
  if (chunk == 0) {
    for (int i = t; i < units; i += kPlanThreads) p.units[i] = tile_of(i);
  } else {
    // units in tile order; the scan carries the units and, above them, the
    // partial slots before each tile
    units = 0;
    int slots = 0;
    for (int base = 0; base < ntiles; base += kPlanThreads) {
      const int i = base + t;
      const int n = i < ntiles ? int(s_n[i]) : 0;
      const int ns = i < ntiles ? max(1, (n + chunk - 1) / chunk) : 0;
      const int mine = ns | (ns > 1 ? ns << 16 : 0);
      int all = 0;
      const int before = block_scan(mine, wsum, &all) - mine;
      if (i < ntiles) {
        PrefillTile x = tile_of(i);
        const int u0 = units + (before & 0xffff), slot0 = slots + (before >> 16);
        for (int s = 0; s < ns; ++s) {
          const unsigned kb = unsigned(s * n / ns), ke = s + 1 < ns ? unsigned((s + 1) * n / ns) : kToEnd;
          x.kt = int(kb | ke << 16);
          x.part = ns > 1 ? ((slot0 + s) << 16 | s << 8 | ns) : 0;
          p.units[u0 + s] = x;
        }
      }
      units += all & 0xffff;
      slots += all >> 16;
      __syncthreads();
    }
    int* counters = reinterpret_cast<int*>(p.ws + p.counters_off[form]);
    for (int i = t; i < slots * p.hkv; i += kPlanThreads) counters[i * kCounterStride] = 0;
  }
  if (t == 0) write_header(p, coarse_tiles, fit, form, units, chunk);
}

struct RunParams {
  const PrefillHeader* header;
  const PrefillTile* tiles;
  const PrefillTile* units;       // (any address where there is no room for them)
  const uint64_t* unit_serial;
  char* parts;
  RunKey key;
  int last_tile, last_unit;       // of the room of either list
  int max_units;                  // that the grid covers
  int tile_bm;                    // positions per coarse tile
  const uint16_t* q;
  int64_t q_st, q_sh;
  int64_t q_ext;  // elements one position's heads span: (heads - 1) * q_sh + head_dim
  const uint16_t* pool;
  unsigned num_pages;  // page ids are 32-bit: capped there
  const int32_t* indices;
  uint16_t* out;
  int64_t o_st, o_sh, o_ext;
  int64_t total_q;
  int hkv, group, causal;
  float scale_log2;
};

typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;
typedef __attribute__((ext_vector_type(4))) short s16x4_t;
typedef __attribute__((ext_vector_type(8))) short s16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4_t;
typedef __attribute__((ext_vector_type(8))) float f32x8_v;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_v;
typedef __attribute__((address_space(3))) char lds_t;

typedef __attribute__((ext_vector_type(2))) unsigned int u32x2_t;

__device__ __forceinline__ void lds_store8(lds_t* p, u32x2_t v) { *(__attribute__((address_space(3))) u32x2_t*)p = v; }
__device__ __forceinline__ u32x4_t lds_load16(const lds_t* p) {
  return *(const __attribute__((address_space(3))) u32x4_t*)p;
}
// gfx950 LDS transpose read: the 16 lanes of a group address 4 rows x 16
// bf16 (lane j: row j/4, elements 4*(j%4)..+3) and lane j receives column j.
__device__ __forceinline__ s16x4_t lds_read_tr16(const lds_t* p) {
  typedef __attribute__((address_space(3))) bf16x4_t lds_v4;
  return __builtin_bit_cast(s16x4_t, __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_v4*)p));
}
// 16 bytes per lane from a buffer straight to LDS: lane l's bytes land at
// dst + 16 l (dst wave-uniform).  The builtin exists for the device pass only
// (the host pass would drop the kernel stubs that reference it).
__device__ __forceinline__ void lds_dma16(__amdgpu_buffer_rsrc_t rs, lds_t* dst, int voffset, int soffset) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)dst, 16, voffset, soffset, 0, 0);
#endif
}
__device__ __forceinline__ float max_xor16(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float max_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ int wave_max_i(int x) {
  for (int o = 32; o > 0; o >>= 1) x = max(x, __shfl_xor(x, o));
  return x;
}
__device__ __forceinline__ float sum_xor16(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float sum_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Slot (16-byte unit of the row) where chunk c of tile row r is staged when
// the rows are unpadded: c XOR a per-row value.  Measured with
// SQ_LDS_BANK_CONFLICT on the Mistral-7B / Qwen2.5-72B head batches (per
// launch): no permutation 70.8M / 210.8M conflict cycles; XOR (r & 15) 6.8M /
// 16.8M; XOR 2 (r & 7) 1.8M / 1.9M (what rows padded by 32 bytes gave), so the 8
// rows of a K read group and the 4 rows x 32 bytes of a V transpose-read
// group land on distinct banks.  128-byte rows (head_dim 64) put two rows in
// a bank period and take XOR 2 ((r >> 1) & 3).
template <int D>
__device__ __forceinline__ int chunk_slot(int r, int c) {
  if constexpr (D == 64) return c ^ (((r >> 1) & 3) << 1);
  else return c ^ ((r & 7) << 1);
}

template <int D, int MAXRB_>
struct PrefillTraits {
  static constexpr int WAVES = waves_for(D);
  static constexpr int THREADS = 64 * WAVES;
  static constexpr int KSTEPS = D / 32;            // 16x16x32 MFMAs per 16-key block of S^T
  static constexpr int NT = D / 16;                // 16-wide head_dim tiles of O
  static constexpr int CPR = D / 8;                // 16-byte chunks per token row
  static constexpr int LOADS = kKvTile * CPR / THREADS;  // 16-byte loads per thread per tile, K and V each
  static_assert(LOADS >= 1 && kKvTile * CPR % THREADS == 0, "tile staging split");
  static constexpr int RS = D * 2;                 // LDS row stride
  static constexpr int TILE = kKvTile * RS;        // bytes of one staged K or V tile
  static constexpr int MAXRB = MAXRB_;             // row blocks per wave
  static constexpr int OUT_BLK = 8 * 32 + kOutPad;  // output staging: bytes per 8 columns
  static constexpr int OB = D / 8 * OUT_BLK;         // output staging: bytes per row block
  // LDS: the double-buffered K / V tiles, reused for the output staging
  static constexpr int SMEM = 2 * 2 * TILE > WAVES * MAXRB * OB ? 2 * 2 * TILE : WAVES * MAXRB * OB;
};

// Normalises row block r of a wave (lane (g, n) holds O rows 4g + i, columns
// 16j + n, and l of row n) and stages it at `ob` for the output stores (see
// the end of the run kernel).
template <int D, int MAXRB>
__device__ __forceinline__ void stage_rows(lds_t* ob, int r, int lane, const mi::f32x4_t (&o)[D / 16], float lt) {
  using T = PrefillTraits<D, MAXRB>;
  const int g = lane >> 4, n = lane & 15;
  const int wcol = n * 32 + (n >> 3) * kOutPad + 8 * g;
  float inv[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float li = mi::lane_shuffle(lt, 4 * g + i);
    inv[i] = li > 0.f ? mi::fast_rcp(li) : 0.f;
  }
#pragma unroll
  for (int j = 0; j < T::NT; ++j)  // column 16j + n: 8-column block 2j + n / 8
    lds_store8(ob + r * T::OB + j * 2 * T::OUT_BLK + wcol,
               u32x2_t{mi::cvt_pk_bf16(o[j][0] * inv[0], o[j][1] * inv[1]),
                       mi::cvt_pk_bf16(o[j][2] * inv[2], o[j][3] * inv[3])});
}

// Where the partials are, and how many slots there are per KV head.
struct PartialArea {
  char* base;
  int slots;
};

// Publishes a split unit's partial (O, m, l in fp32) and counts it; the last
// of the tile's units reads all of them back in split order (so the result
// does not depend on which came last), stages the merged rows for the output
// stores and returns true.  The others return false.  Partials go through
// device-coherent (sc1) stores and loads, as the units of a tile may run on
// different XCDs; the counter is back at zero for the next run of the plan.
// What bounds a merge is the round trip of its reads (104 KB per split at
// head_dim 128): the wave walks (row block, split) as one sequence with DP
// row blocks on their way (four of them at head_dim 64 would take the whole
// kernel from four waves per SIMD to three).
template <int D, int MAXRB>
__device__ __forceinline__ bool merge_splits(const RunParams& p, int part, const PartialArea& pa, int hkv, int w, int lane, int nblk,
                                             lds_t* lds, lds_t* ob, const mi::f32x4_t (&o)[MAXRB][D / 16],
                                             const float (&m_run)[MAXRB], const float (&lt)[MAXRB]) {
  using T = PrefillTraits<D, MAXRB>;
  constexpr int NT = T::NT;
  constexpr int CP = 16;  // cache policy: sc1 (device scope)
  constexpr int DP = D == 256 ? 1 : MAXRB == 3 || D == 64 ? 3 : 4;
  constexpr int WB = MAXRB * (NT * 1024 + 512);  // bytes of one wave's partial
  static_assert(WB * T::WAVES == int(partial_bytes(D, MAXRB)), "partial layout");
  const int g = lane >> 4;
  const int nsplit = part & 0xff, split = (part >> 8) & 0xff, slot0 = int(unsigned(part) >> 16) - split;
  char* base = pa.base;
  const int nslots = pa.slots;
  // the wave's partial of split s, one descriptor each: the slots of one tile
  // and KV head lie hkv slots apart
  auto rsrc = [&](int s) {
    char* a = base + (int64_t(slot0 + s) * p.hkv + hkv) * int64_t(WB * T::WAVES) + w * WB;
    return __builtin_amdgcn_make_buffer_rsrc(a, (short)0, WB, kBufferWord3);
  };
  {
    const __amdgpu_buffer_rsrc_t rs = rsrc(split);
#pragma unroll
    for (int r = 0; r < MAXRB; ++r) {
      if (r >= nblk) continue;
#pragma unroll
      for (int j = 0; j < NT; ++j)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, o[r][j]), rs, lane * 16, (r * NT + j) * 1024, CP);
      __builtin_amdgcn_raw_buffer_store_b64(u32x2_t{__float_as_uint(m_run[r]), __float_as_uint(lt[r])}, rs, lane * 8,
                                            MAXRB * NT * 1024 + r * 512, CP);
    }
  }
  // every wave's stores are acknowledged before one lane counts the unit
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
  __syncthreads();
  int* counter = reinterpret_cast<int*>(base + int64_t(nslots) * p.hkv * int64_t(WB * T::WAVES)) +
                 (int64_t(slot0) * p.hkv + hkv) * kCounterStride;
  __attribute__((address_space(3))) int* flag = (__attribute__((address_space(3))) int*)lds;
  if (threadIdx.x == 0) *flag = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const int prev = __builtin_amdgcn_readfirstlane(*flag);
  __syncthreads();  // the flag's bytes are staged over below
  if (prev != nsplit - 1) return false;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  if (threadIdx.x == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

  u32x4_t v[DP][NT];
  u32x2_t ml[DP];
  const int steps = nblk * nsplit;
  int rl = 0, sl = 0;  // the next step to load
  auto load = [&](int q) {
    const __amdgpu_buffer_rsrc_t rs = rsrc(sl);
    ml[q] = __builtin_amdgcn_raw_buffer_load_b64(rs, lane * 8, MAXRB * NT * 1024 + rl * 512, CP);
#pragma unroll
    for (int j = 0; j < NT; ++j)
      v[q][j] = __builtin_amdgcn_raw_buffer_load_b128(rs, lane * 16, (rl * NT + j) * 1024, CP);
    if (++sl == nsplit) {
      sl = 0;
      ++rl;
    }
  };
#pragma unroll
  for (int q = 0; q < DP; ++q)
    if (q < steps) load(q);
  mi::f32x4_t acc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) acc[j] = mi::f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  int r = 0, s = 0;
  for (int k = 0; k < steps; k += DP) {
#pragma unroll
    for (int q = 0; q < DP; ++q) {
      if (k + q >= steps) break;
      // row n of the block: the weights of what is merged so far and of this
      // split (0 for a split that saw no key of the row: its m is -inf)
      const float ms = __uint_as_float(ml[q].x), ls = __uint_as_float(ml[q].y);
      const float mn = fmaxf(m, ms);
      const float f0 = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mn);
      const float f1 = ms == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms - mn);
      m = mn;
      l = l * f0 + ls * f1;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float a0 = mi::lane_shuffle(f0, 4 * g + i), a1 = mi::lane_shuffle(f1, 4 * g + i);
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[j][i] = acc[j][i] * a0 + __uint_as_float(v[q][j][i]) * a1;
      }
      if (k + q + DP < steps) load(q);
      if (++s == nsplit) {
        stage_rows<D, MAXRB>(ob, r, lane, acc, l);
        m = -INFINITY;
        l = 0.f;
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[j] = mi::f32x4_t{0.f, 0.f, 0.f, 0.f};
        s = 0;
        ++r;
      }
    }
  }
  return true;
}

// One unit of the run (a workgroup), MAXRB row blocks per wave.
template <int D, int MAXRB>
__device__ __forceinline__ void run_unit(const RunParams& p, const PrefillTile& t, const PartialArea& pa, int hkv, int bm,
                                         lds_t* lds) {
  using T = PrefillTraits<D, MAXRB>;
  const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  const int g = lane >> 4, n = lane & 15;
  const int off = t.kv_len - t.qo_len;
  // the workgroup's rows in position-major order: row R is position R / group
  // of the tile, head R % group of this KV head's group; row block rb holds
  // rows 16 rb .. 16 rb + 15
  const int nrows = bm * p.group;
  const int nrb = (nrows + 15) / 16;

  // ---- this wave's row blocks: rb = w, w + 4
  mi::bf16x8_t qb[T::MAXRB][T::KSTEPS];
  mi::f32x4_t o[T::MAXRB][T::NT];
  float m_run[T::MAXRB], l_run[T::MAXRB];
  int qpos[T::MAXRB];     // request-relative position of this lane's row n (-1: none)
  int lim[T::MAXRB];      // last key this lane's row may see (-1: none)
  int rb_hi[T::MAXRB];    // keys this row block needs (causal)
  int head[T::MAXRB];     // this lane's row's Q head
  int lpos[T::MAXRB];     // this lane's row's position within the tile (-1: none)
  int nblk = 0;
  const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.q + int64_t(t.q_begin) * p.q_st), (short)0,
      int((int64_t(max(t.q_rows, 1) - 1) * p.q_st + p.q_ext) * 2), kBufferWord3);
#pragma unroll
  for (int r = 0; r < T::MAXRB; ++r) {
    const int rb = w + T::WAVES * r;
    const bool has = rb < nrb;
    nblk += has ? 1 : 0;
    const int row = rb * 16 + n;
    const int local = row / p.group;
    head[r] = hkv * p.group + (row - local * p.group);
    const bool valid = has && row < nrows && local < t.q_rows;
    lpos[r] = valid ? local : -1;
    qpos[r] = valid ? t.row0 + local : -1;
    lim[r] = !valid ? -1 : (p.causal ? min(t.kv_len - 1, qpos[r] + off) : t.kv_len - 1);
    const int last = t.row0 + min((rb * 16 + 15) / p.group, t.q_rows - 1);  // the block's last position
    rb_hi[r] = !has ? 0 : (p.causal ? min(t.kv_len, last + off + 1) : t.kv_len);
    // Q rows through a descriptor over the tile's rows: a row past the tile
    // reads out of range (zeros), so the loads are unconditional
    const int qoff = valid ? int((int64_t(local) * p.q_st + int64_t(head[r]) * p.q_sh + g * 8) * 2) : 0x7ffffff0;
#pragma unroll
    for (int s = 0; s < T::KSTEPS; ++s)
      qb[r][s] = __builtin_bit_cast(mi::bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(rq, qoff, s * 64, 0));
#pragma unroll
    for (int j = 0; j < T::NT; ++j) o[r][j] = mi::f32x4_t{0.f, 0.f, 0.f, 0.f};
    m_run[r] = -INFINITY;
    l_run[r] = 0.f;
  }
  // smallest valid row position of the wave (for the unmasked-tile test)
  int qmin = 0x7fffffff;
#pragma unroll
  for (int r = 0; r < T::MAXRB; ++r)
    if (qpos[r] >= 0) qmin = min(qmin, qpos[r]);
  qmin = __builtin_amdgcn_readfirstlane(-wave_max_i(-qmin));
  int block_hi = p.causal ? min(t.kv_len, t.row0 + t.q_rows + off) : t.kv_len;
  block_hi = max(block_hi, 0);
  // this unit's KV tiles (a split tile's last unit takes all that remain)
  const int nsplit = t.part & 0xff;
  const int ntile = __builtin_amdgcn_readfirstlane(min((block_hi + kKvTile - 1) / kKvTile,
      unsigned(t.kt) >> 16 == kToEnd ? 0x7fffffff : int(unsigned(t.kt) >> 16)));
  const int kt0 = t.kt & 0xffff;

  // ---- staging.  A load of a wave covers whole rows of one page (1 KB <= 16
  // rows), so the page id is wave-uniform -- a
  // scalar load, fetched one tile ahead -- and each page gets a buffer
  // descriptor (size 0 past the request's pages; on the request's last page
  // the size stops after its valid V rows, so the V rows past kv_len read as
  // zeros: P is 0 there, but 0 * NaN would poison the MFMA).  No address
  // arithmetic or branches per load.
  const int tok_bytes = p.hkv * D * 2;
  const int kv_bytes = kPageSize * tok_bytes;
  const int page_bytes = 2 * kv_bytes;
  const int npages_req = (t.kv_len + kPageSize - 1) / kPageSize;
  const int last_rows = t.kv_len - (npages_req - 1) * kPageSize;
  int voff[T::LOADS], pit[T::LOADS];
  // Load i of wave w fills 1 KB block b = WAVES i + w of the tile: RPB rows,
  // lane l taking row b RPB + l / CPR and slot l % CPR of it, i.e. the chunk
  // chunk_slot(row, slot) (the permutation is its own inverse); a block lies
  // inside one page, so the page index is wave-uniform.
  constexpr int RPB = 1024 / (D * 2);
#pragma unroll
  for (int i = 0; i < T::LOADS; ++i) {
    const int bk = T::WAVES * i + w;
    const int tr = bk * RPB + lane / T::CPR;
    pit[i] = __builtin_amdgcn_readfirstlane(bk * RPB / kPageSize);
    voff[i] = (tr % kPageSize) * tok_bytes + hkv * D * 2 + chunk_slot<D>(tr, lane % T::CPR) * 16;
  }
  int pid[T::LOADS];
  // page ids through the constant address space: a uniform index then
  // compiles to a scalar load (kv_indices is not written during the launch)
  typedef __attribute__((address_space(4))) const int32_t const_i32;
  const const_i32* kv_ids = (const const_i32*)(p.indices);
  auto fetch_ids = [&](int kt) {
#pragma unroll
    for (int i = 0; i < T::LOADS; ++i) {
      const int pg_idx = kt * (kKvTile / kPageSize) + pit[i];
      // clamped into the request's pages (it has >= 1 page whenever there is
      // a tile); an id past the end is dropped when it is used, so that
      // nothing here waits for these loads (with the test beside them each of
      // the loads was waited for in turn)
      pid[i] = kv_ids[t.kv_page_begin + min(pg_idx, npages_req - 1)];
    }
  };
  auto load_tile = [&](int kt, int buf) {
#pragma unroll
    for (int i = 0; i < T::LOADS; ++i) {
      const int pg = __builtin_amdgcn_readfirstlane(pid[i]);
      const int pg_idx = kt * (kKvTile / kPageSize) + pit[i];
      const bool ok = unsigned(pg) < p.num_pages && pg_idx < npages_req;
      const int size = !ok ? 0 : (pg_idx == npages_req - 1 ? kv_bytes + last_rows * tok_bytes : page_bytes);
      const char* base = reinterpret_cast<const char*>(p.pool) + (ok ? int64_t(pg) * page_bytes : 0);
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, size, kBufferWord3);
      lds_t* kdst = lds + buf * 2 * T::TILE + 1024 * (T::WAVES * i + w);
      lds_dma16(rs, kdst, voff[i], 0);
      lds_dma16(rs, kdst + T::TILE, voff[i], kv_bytes);
    }
  };
  if (kt0 < ntile) {
    fetch_ids(kt0);
    load_tile(kt0, 0);
    fetch_ids(kt0 + 1);
  }
  // Everything loaded so far (Q, tile 0, the next page ids) is waited for
  // here, so the loop head carries no pending load from before the loop;
  // without it the compiler put a full vmcnt(0) before the first score MFMA
  // of every tile, which also waited for the next tile's prefetch.
  __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
  __syncthreads();

  // LDS read offsets inside a staged tile: K row kb 16 + n (chunk 4 s + g) for
  // the score operand, V rows 4 g + n / 4 (bytes 32 j + 8 (n & 3)) for the
  // transpose reads; tile rows are r and r + 16 k, whose permutation depends
  // on r % 16 only.
  int koff[T::KSTEPS], voff_lds[T::NT];
#pragma unroll
  for (int s2 = 0; s2 < T::KSTEPS; ++s2)
    koff[s2] = n * T::RS + chunk_slot<D>(n, 4 * s2 + g) * 16;
#pragma unroll
  for (int j = 0; j < T::NT; ++j) {
    const int vr = 4 * g + (n >> 2);
    voff_lds[j] = vr * T::RS + chunk_slot<D>(vr, 2 * j + ((n & 3) >> 1)) * 16 + (n & 1) * 8;
  }

  for (int kt = kt0; kt < ntile; ++kt) {
    const int buf = (kt - kt0) & 1;
    if (kt + 1 < ntile) {
      load_tile(kt + 1, buf ^ 1);
      fetch_ids(kt + 2);
    }
    const int kv0 = kt * kKvTile;
    const lds_t* kl = lds + buf * 2 * T::TILE;
    const lds_t* vl = kl + T::TILE;
    // All of the wave's row blocks are computed together so each K / V
    // operand read from LDS feeds MAXRB MFMAs.  A block with nothing left to
    // do (causally finished, or absent: qpos = -1) masks every key and adds
    // exactly zero, so no per-block branches are needed.
    bool any = false;
#pragma unroll
    for (int r = 0; r < T::MAXRB; ++r) any = any || (r < nblk && kv0 < rb_hi[r]);
    if (any) {
      // No key of the tile needs a mask: all are < kv_len and (causal) visible
      // to the wave's first valid row.  (Rows past the tile's end hold zero
      // queries and are never written, so they need no mask either.)
      const bool full = kv0 + kKvTile <= t.kv_len && (!p.causal || kv0 + kKvTile - 1 <= qmin + off);
      // ---- one tile: S^T for the four 16-key blocks (raw scores; the softmax
      // scale is applied inside the exponent; two copies of the score loop,
      // so full tiles carry no mask code), the row maxima, one lazy-rescale
      // branch for the wave, then exp / pack / P V half by half, so the P V
      // MFMAs of keys 0-31 can overlap the exponentials of keys 32-63.
      float sv[T::MAXRB][kKvTile / 16][4];
      auto scores = [&](auto masked) {
#pragma unroll
        for (int kb = 0; kb < kKvTile / 16; ++kb) {
          mi::bf16x8_t ka[T::KSTEPS];
#pragma unroll
          for (int s = 0; s < T::KSTEPS; ++s)
            ka[s] = __builtin_bit_cast(mi::bf16x8_t, lds_load16(kl + kb * 16 * T::RS + koff[s]));
#pragma unroll
          for (int r = 0; r < T::MAXRB; ++r) {
            mi::f32x4_t c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < T::KSTEPS; ++s) c = mi::mfma_16x16x32_bf16(ka[s], qb[r][s], c);
#pragma unroll
            for (int i = 0; i < 4; ++i) sv[r][kb][i] = c[i];
            if constexpr (decltype(masked)::value) {
              // key kv0 + kb*16 + 4g + i is visible iff kb*16 + i <= lim - kv0 - 4g
              const int rel = lim[r] - kv0 - 4 * g;
#pragma unroll
              for (int i = 0; i < 4; ++i)
                if (kb * 16 + i > rel) sv[r][kb][i] = -INFINITY;
            }
          }
        }
      };
      // The score MFMAs and the row maxima run at raised wave priority: the
      // other workgroup's wave on the SIMD is then usually in its softmax /
      // P V part, and the arbiter issues this wave's MFMAs first while that
      // VALU work fills the gaps (Qwen2.5-72B / Qwen2.5-7B head batches
      // -1.9..-2.2 / -1.1..-1.5 % over three boxes, Mistral-7B heads
      // -1.2..+0.9 %; around the P V MFMAs as well: no better; the reverse
      // -- priority over the softmax instead -- gains the same: what helps is
      // that the two workgroups' waves on a SIMD stop moving in step)
      __builtin_amdgcn_s_setprio(1);
      if (full) scores(std::false_type{});
      else scores(std::true_type{});
      {
        float mloc[T::MAXRB];
        bool need[T::MAXRB];
        bool any_need = false;
#pragma unroll
        for (int r = 0; r < T::MAXRB; ++r) {
          float m = sv[r][0][0];
#pragma unroll
          for (int kb = 0; kb < kKvTile / 16; ++kb)
#pragma unroll
            for (int i = 0; i < 4; ++i) m = fmaxf(m, sv[r][kb][i]);
          mloc[r] = max_xor32(max_xor16(m)) * p.scale_log2;  // scale > 0 keeps the arg max
          need[r] = mloc[r] > m_run[r] + kLazyRescale;
          any_need = any_need || need[r];
        }
        __builtin_amdgcn_s_setprio(0);
        if (__builtin_amdgcn_ballot_w64(any_need)) {
#pragma unroll
          for (int r = 0; r < T::MAXRB; ++r) {
            // a row that has seen no key yet (m_run = -inf) still has O = 0
            // and l = 0: only its max moves, nothing is rescaled
            const bool scale = need[r] && m_run[r] != -INFINITY;
            const float f = scale ? __builtin_amdgcn_exp2f(m_run[r] - mloc[r]) : 1.f;
            m_run[r] = need[r] ? mloc[r] : m_run[r];
            l_run[r] *= f;
            if (__builtin_amdgcn_ballot_w64(scale)) {
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const float fo = mi::lane_shuffle(f, 4 * g + i);
#pragma unroll
                for (int j = 0; j < T::NT; ++j) o[r][j][i] *= fo;
              }
            }
          }
        }
#pragma unroll
        for (int h = 0; h < kKvTile / 32; ++h) {
          // exp2(-inf - m) = 0 for masked keys; m is taken as 0 while the row
          // has seen no key (m_run still -inf), avoiding -inf - -inf
          mi::bf16x8_t pa[T::MAXRB];
#pragma unroll
          for (int r = 0; r < T::MAXRB; ++r) {
            const float m_use = (m_run[r] == -INFINITY) ? 0.f : m_run[r];
            float pv[2][4];
            float ps = 0.f;
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                pv[kk][i] = __builtin_amdgcn_exp2f(fmaf(sv[r][2 * h + kk][i], p.scale_log2, -m_use));
                ps += pv[kk][i];
              }
            l_run[r] += ps;
            pa[r] = __builtin_bit_cast(
                mi::bf16x8_t, __builtin_convertvector((f32x8_v){pv[0][0], pv[0][1], pv[0][2], pv[0][3], pv[1][0],
                                                                pv[1][1], pv[1][2], pv[1][3]},
                                                      bf16x8_v));
          }
          // ---- O += P V over key blocks (2h, 2h + 1)
          const lds_t* v0 = vl + 2 * h * 16 * T::RS;
          // The transpose reads go through inline asm here: with the builtin the
          // compiler waited for every load to LDS in flight (the next tile's)
          // before the first of them.  One statement per group of 4 columns:
          // 8 reads (the second page's rows 16 * RS further) and the wait for
          // them, so its outputs hold the data when it ends.
          static_assert(T::NT % 4 == 0, "column groups of 4");
          const uint32_t vb0 = uint32_t(reinterpret_cast<uintptr_t>(v0));
#pragma unroll
          for (int q = 0; q < T::NT / 4; ++q) {
            const int j0 = 4 * q;
            u32x2_t ra[4], rb[4];
            asm volatile(
                "ds_read_b64_tr_b16 %0, %8\n\t"
                "ds_read_b64_tr_b16 %1, %8 offset:%12\n\t"
                "ds_read_b64_tr_b16 %2, %9\n\t"
                "ds_read_b64_tr_b16 %3, %9 offset:%12\n\t"
                "ds_read_b64_tr_b16 %4, %10\n\t"
                "ds_read_b64_tr_b16 %5, %10 offset:%12\n\t"
                "ds_read_b64_tr_b16 %6, %11\n\t"
                "ds_read_b64_tr_b16 %7, %11 offset:%12\n\t"
                "s_waitcnt lgkmcnt(0)"
                : "=&v"(ra[0]), "=&v"(rb[0]), "=&v"(ra[1]), "=&v"(rb[1]), "=&v"(ra[2]), "=&v"(rb[2]), "=&v"(ra[3]),
                  "=&v"(rb[3])
                : "v"(vb0 + voff_lds[j0]), "v"(vb0 + voff_lds[j0 + 1]), "v"(vb0 + voff_lds[j0 + 2]),
                  "v"(vb0 + voff_lds[j0 + 3]), "i"(16 * T::RS)
                : "memory");
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
              const mi::bf16x8_t vb =
                  __builtin_bit_cast(mi::bf16x8_t, u32x4_t{ra[jj].x, ra[jj].y, rb[jj].x, rb[jj].y});
#pragma unroll
              for (int r = 0; r < T::MAXRB; ++r) o[r][j0 + jj] = mi::mfma_16x16x32_bf16(pa[r], vb, o[r][j0 + jj]);
            }
          }
        }
      }
    }
    // the next tile's rows are in LDS (the loads went straight there)
    if (kt + 1 < ntile) __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
    __syncthreads();
  }

  // ---- normalise and store.  Lane (g, n) holds O rows 4g + i, columns 16j + n.
  // The normalised rows go through LDS (the K / V buffers are free after the
  // loop's last barrier) as a column-major block per row block: element
  // (row, col) at byte col * 32 + (col / 8) * kOutPad + row * 2, so a lane's
  // four rows of one column are one 8-byte write, and the LDS transpose read
  // of a 4-column x 16-row block hands lane n four consecutive columns of row
  // n: two reads give 16 contiguous bytes of an output row, one 16-byte store
  // through a descriptor over the tile's output rows (rows past the tile get
  // an out-of-range offset, so the stores are unconditional).
  constexpr int kOutBlk = T::OUT_BLK;
  constexpr int OB = T::OB;
  lds_t* const ob = lds + w * T::MAXRB * OB;
  float lt[T::MAXRB];
#pragma unroll
  for (int r = 0; r < T::MAXRB; ++r) lt[r] = sum_xor32(sum_xor16(l_run[r]));
  // Every unit stages its own rows first, a split one for nothing: `o` is then
  // dead once a partial is published, whichever way the unit goes on, and the
  // merge has its registers for reads in flight.
#pragma unroll
  for (int r = 0; r < T::MAXRB; ++r)
    if (r < nblk) stage_rows<D, MAXRB>(ob, r, lane, o[r], lt[r]);
  if (nsplit > 1 && !merge_splits<D, MAXRB>(p, t.part, pa, hkv, w, lane, nblk, lds, ob, o, m_run, lt))
    return;
  __syncthreads();
  const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.out + int64_t(t.q_begin) * p.o_st), (short)0,
      int((int64_t(max(t.q_rows, 1) - 1) * p.o_st + p.o_ext) * 2), kBufferWord3);
  // lane (g, n) reads columns 32q + 8g + [0, 8) of row n
  const int rcol = g * kOutBlk + (n >> 2) * 32 + (n & 3) * 8;
#pragma unroll
  for (int r = 0; r < T::MAXRB; ++r) {
    if (r >= nblk) continue;
    const int local = lpos[r];
    const bool valid = local >= 0 && t.q_begin + local < p.total_q;
    const int off = valid ? int((int64_t(local) * p.o_st + int64_t(head[r]) * p.o_sh) * 2) + 16 * g : 0x7ffffff0;
#pragma unroll
    for (int q = 0; q < D / 32; ++q) {
      const lds_t* src = ob + r * OB + q * 4 * kOutBlk + rcol;
      const s16x4_t a = lds_read_tr16(src), c = lds_read_tr16(src + 128);
      __builtin_amdgcn_raw_buffer_store_b128(
          __builtin_bit_cast(u32x4_t, (s16x8_t){a[0], a[1], a[2], a[3], c[0], c[1], c[2], c[3]}), ro, off, 64 * q, 0);
    }
  }
}

// Waves per SIMD of the run.  head_dim 64 keeps four (125 registers): with three,
// 832 tiles of short prompts took 9.3 us instead of 7.3.
constexpr int run_waves(int head_dim) { return head_dim == 64 ? 4 : head_dim == 128 ? 2 : 1; }

// The units of the plan if this run may take them, else its tiles.  The plan
// says which form the units have: coarse, RB row blocks per wave, or fine, one.
template <int D, int RB>
__global__ __launch_bounds__(64 * waves_for(D)) __attribute__((amdgpu_waves_per_eu(run_waves(D)))) void prefill_run_kernel(RunParams p) {
  __shared__ __attribute__((aligned(16))) char smem[PrefillTraits<D, RB>::SMEM];  // [buffer][K, V], then the output rows
  static_assert(PrefillTraits<D, 1>::SMEM <= PrefillTraits<D, RB>::SMEM, "LDS of the fine form");
  lds_t* lds = (lds_t*)smem;
  // every argument from the argument segment at once: left to the compiler, some of
  // these reads came after the header's, one more round trip each
  __asm__ volatile("" ::"s"(p.header), "s"(p.tiles), "s"(p.units), "s"(p.unit_serial), "s"(p.parts), "s"(p.key.ws),
                   "s"(p.key.bytes), "s"(p.key.stream), "s"(p.key.shape), "s"(p.last_tile), "s"(p.last_unit),
                   "s"(p.max_units), "s"(p.tile_bm), "s"(p.q), "s"(p.q_st), "s"(p.q_sh), "s"(p.q_ext), "s"(p.pool),
                   "s"(p.num_pages), "s"(p.indices), "s"(p.total_q), "s"(p.hkv), "s"(p.group), "s"(p.causal),
                   "s"(p.scale_log2));
  const int tile_idx = int(blockIdx.x) / p.hkv;
  const int hkv = int(blockIdx.x) - tile_idx * p.hkv;
  // The header and the record (not written during the launch) are read through
  // the constant address space, so they arrive in scalar registers: as vector
  // loads, which the stores of partials otherwise make of them, the compiler
  // put a per-lane loop around every page load of head_dim 256 (2.9 -> 3.3 us
  // per KV tile).
  typedef __attribute__((address_space(4))) const PrefillHeader const_header;
  typedef __attribute__((address_space(4))) const int const_int;
  const const_header* h = (const const_header*)(p.header);
  typedef __attribute__((address_space(4))) const uint64_t const_u64;
  // Both lists' records (clamped into them) go out with the header, and the tests
  // have no branches, so that all of it takes one round trip.
  const const_int* fu = (const const_int*)(p.units + min(tile_idx, p.last_unit));
  const const_int* ft = (const const_int*)(p.tiles + min(tile_idx, p.last_tile));
  const PrefillTile tu{fu[0], fu[1], fu[2], fu[3], fu[4], fu[5], fu[6], fu[7]};
  const PrefillTile tt{ft[0], ft[1], ft[2], ft[3], ft[4], ft[5], ft[6], ft[7]};
  const uint64_t serial = *(const const_u64*)(p.unit_serial);
  const int num_units = h->units, num_tiles = h->num_tiles, unit_bm = h->bm, blocks = h->row_blocks;
  const uint64_t differs = (h->key.ws ^ p.key.ws) | (h->key.bytes ^ p.key.bytes) | (h->key.stream ^ p.key.stream) |
                           (h->key.shape ^ p.key.shape) | (h->serial ^ serial) | uint64_t(p.key.stream == 0);
  const PartialArea pa{p.parts, h->slots};
  const bool own = (num_units > 0) & (differs == 0) & (num_units <= p.max_units);
  const PrefillTile t{own ? tu.q_begin : tt.q_begin, own ? tu.q_rows : tt.q_rows, own ? tu.qo_len : tt.qo_len,
                      own ? tu.kv_len : tt.kv_len,   own ? tu.row0 : tt.row0,     own ? tu.kv_page_begin : tt.kv_page_begin,
                      own ? tu.kt : tt.kt,           own ? tu.part : tt.part};
  __asm__ volatile("" ::"s"(t.q_begin), "s"(t.q_rows), "s"(t.qo_len), "s"(t.kv_len), "s"(t.row0), "s"(t.kv_page_begin),
                   "s"(t.kt), "s"(t.part), "s"(unit_bm), "s"(blocks), "s"(pa.slots));  // (else their loads sink below the return)
  if (tile_idx >= (own ? num_units : num_tiles)) return;  // whole workgroup
  const int bm = own ? unit_bm : p.tile_bm;
  if (RB > 1 && own && blocks == 1) run_unit<D, 1>(p, t, pa, hkv, bm, lds);
  else run_unit<D, RB>(p, t, pa, hkv, bm, lds);
}

}  // namespace

extern "C" size_t mi_prefill_workspace_size(int32_t batch_size, int64_t total_q) {
  if (batch_size < 0 || total_q < 0) return 0;
  return prefill_ws_bytes(batch_size, total_q);
}

extern "C" int mi_prefill_plan(void* workspace, size_t workspace_bytes, const int32_t* qo_indptr,
                               const int32_t* kv_indptr, const int32_t* kv_last_page_len,
                               int32_t batch_size, int64_t total_q, int32_t num_qo_heads,
                               int32_t num_kv_heads, int32_t head_dim, int32_t page_size,
                               mi_stream_t stream) {
  mi::clear_error();
  if (batch_size < 0 || total_q < 0) return mi::fail(MI_ERR_INVALID, "prefill plan: negative sizes");
  if (num_qo_heads <= 0 || num_kv_heads <= 0 || num_qo_heads % num_kv_heads)
    return mi::fail(MI_ERR_INVALID, "prefill plan: bad head counts (%d, %d)", num_qo_heads, num_kv_heads);
  if (num_qo_heads / num_kv_heads > 8)
    return mi::fail(MI_ERR_UNSUPPORTED, "prefill plan: group %d (built for 1..8)", num_qo_heads / num_kv_heads);
  if (page_size != kPageSize) return mi::fail(MI_ERR_UNSUPPORTED, "prefill plan: page_size %d (built for 16)", page_size);
  const size_t need = prefill_ws_bytes(batch_size, total_q);
  if (!workspace || workspace_bytes < need)
    return mi::fail(MI_ERR_WORKSPACE, "prefill plan: workspace %zu bytes, need %zu", workspace_bytes, need);
  if (batch_size > 0 && (!qo_indptr || !kv_indptr || !kv_last_page_len))
    return mi::fail(MI_ERR_INVALID, "prefill plan: null indptr argument");
  char* ws = static_cast<char*>(workspace);
  PlanParams pp;
  pp.qo_indptr = qo_indptr;
  pp.kv_indptr = kv_indptr;
  pp.last_page_len = kv_last_page_len;
  pp.batch = batch_size;
  pp.capacity = int(tile_capacity(batch_size, total_q));
  pp.group = num_qo_heads / num_kv_heads;
  pp.hkv = num_kv_heads;
  const int cus = mi::num_cus();
  pp.resident = resident_groups(cus, head_dim);
  pp.cus = head_dim == 256 ? 0 : cus;
  const UnitLayout L = unit_layout(pp.resident, workspace_bytes, num_kv_heads, head_dim);
  static std::atomic<uint64_t> plans{0};
  pp.serial = (plans.fetch_add(1, std::memory_order_relaxed) + 1) * 0x9e3779b97f4a7c15ull;
  pp.key = run_key(workspace, workspace_bytes, num_kv_heads, pp.group, head_dim, static_cast<hipStream_t>(stream));
  pp.unit_capacity = pp.key.stream ? L.capacity : 0;
  pp.tile_room = L.capacity ? int(std::min<size_t>((L.off - 256) / sizeof(PrefillTile), 1 << 30)) : 0;
  for (int form = 0; form < 2; ++form) {
    pp.blocks[form] = form ? row_blocks(head_dim) : 1;
    pp.bm[form] = rows_per_tile(pp.group, head_dim, pp.blocks[form]);
    pp.slots[form] = form ? L.coarse : L.fine;
    pp.counters_off[form] = L.parts + size_t(pp.slots[form]) * num_kv_heads * partial_bytes(head_dim, pp.blocks[form]);
  }
  pp.ws = ws;
  pp.header = reinterpret_cast<PrefillHeader*>(ws);
  pp.tiles = reinterpret_cast<PrefillTile*>(ws + 256);
  pp.unit_serial = reinterpret_cast<uint64_t*>(ws + L.off);
  pp.units = reinterpret_cast<PrefillTile*>(ws + L.off + 256);
  hipLaunchKernelGGL(prefill_plan_kernel, dim3(1), dim3(kPlanThreads), 0, static_cast<hipStream_t>(stream), pp);
  return mi::check_launch("prefill_plan_kernel");
}

extern "C" int mi_prefill_run(void* workspace, size_t workspace_bytes, const void* q,
                              int64_t q_stride_token, int64_t q_stride_head, const void* paged_kv_cache,
                              int64_t num_pages, const int32_t* kv_indices, void* out,
                              int64_t out_stride_token, int64_t out_stride_head, int32_t batch_size,
                              int64_t total_q, int32_t num_qo_heads, int32_t num_kv_heads,
                              int32_t head_dim, int32_t page_size, int32_t causal, float sm_scale,
                              mi_stream_t stream) {
  mi::clear_error();
  if (batch_size < 0 || total_q < 0 || num_qo_heads <= 0 || num_kv_heads <= 0 || num_qo_heads % num_kv_heads)
    return mi::fail(MI_ERR_INVALID, "prefill run: bad sizes");
  if (num_qo_heads / num_kv_heads > 8)
    return mi::fail(MI_ERR_UNSUPPORTED, "prefill run: group %d (built for 1..8)", num_qo_heads / num_kv_heads);
  if (page_size != kPageSize) return mi::fail(MI_ERR_UNSUPPORTED, "prefill run: page_size %d (built for 16)", page_size);
  if (head_dim != 64 && head_dim != 128 && head_dim != 256)
    return mi::fail(MI_ERR_UNSUPPORTED, "prefill run: head_dim %d (built for 64, 128, 256)", head_dim);
  const size_t need = prefill_ws_bytes(batch_size, total_q);
  if (!workspace || workspace_bytes < need)
    return mi::fail(MI_ERR_WORKSPACE, "prefill run: workspace %zu bytes, need %zu", workspace_bytes, need);
  if (total_q == 0 || batch_size == 0) return MI_OK;
  if (!q || !paged_kv_cache || !kv_indices || !out) return mi::fail(MI_ERR_INVALID, "prefill run: null pointer");
  if ((reinterpret_cast<uintptr_t>(q) & 15) || (reinterpret_cast<uintptr_t>(paged_kv_cache) & 15) ||
      (reinterpret_cast<uintptr_t>(out) & 15) || q_stride_token % 8 || q_stride_head % 8 ||
      out_stride_token % 8 || out_stride_head % 8)
    return mi::fail(MI_ERR_INVALID, "prefill run: q rows, out rows and pool must be 16-byte aligned");
  if (q_stride_token < 0 || q_stride_head < 0 || out_stride_token < 0 || out_stride_head < 0)
    return mi::fail(MI_ERR_INVALID, "prefill run: negative stride");
  const int resident = resident_groups(mi::num_cus(), head_dim);
  const int64_t grid = run_groups(resident, batch_size, total_q, num_qo_heads / num_kv_heads, num_kv_heads, head_dim);
  if (grid > 0x7fffffff) return mi::fail(MI_ERR_INVALID, "prefill run: too many tiles");
  char* ws = static_cast<char*>(workspace);
  RunParams rp;
  rp.header = reinterpret_cast<const PrefillHeader*>(ws);
  rp.tiles = reinterpret_cast<const PrefillTile*>(ws + 256);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const UnitLayout L = unit_layout(resident, workspace_bytes, num_kv_heads, head_dim);
  rp.unit_serial = reinterpret_cast<const uint64_t*>(ws + L.off);
  rp.units = reinterpret_cast<const PrefillTile*>(ws + L.off + 256);
  rp.parts = ws + L.parts;
  rp.last_tile = int(std::min<size_t>(tile_capacity(batch_size, total_q), 1 << 30)) - 1;
  rp.last_unit = std::max(L.capacity, 1) - 1;
  rp.max_units = int(grid / num_kv_heads);
  rp.key = run_key(workspace, workspace_bytes, num_kv_heads, num_qo_heads / num_kv_heads, head_dim, s);
  rp.q = static_cast<const uint16_t*>(q);
  rp.q_st = q_stride_token;
  rp.q_sh = q_stride_head;
  rp.pool = static_cast<const uint16_t*>(paged_kv_cache);
  rp.num_pages = unsigned(std::min<int64_t>(std::max<int64_t>(num_pages, 0), 0x7fffffff));
  rp.indices = kv_indices;
  rp.out = static_cast<uint16_t*>(out);
  rp.o_st = out_stride_token;
  rp.o_sh = out_stride_head;
  rp.total_q = total_q;
  rp.hkv = num_kv_heads;
  rp.group = num_qo_heads / num_kv_heads;
  rp.causal = causal ? 1 : 0;
  const int bm = rp.tile_bm = rows_per_tile(rp.group, head_dim, row_blocks(head_dim));
  // a tile addresses its q / out rows through one buffer descriptor each, by
  // 32-bit byte offsets from its first position: any strides (heads inside a
  // position's row, or head-major) whose tile extent fits
  rp.q_ext = int64_t(num_qo_heads - 1) * q_stride_head + head_dim;
  rp.o_ext = int64_t(num_qo_heads - 1) * out_stride_head + head_dim;
  const int64_t q_span = (int64_t(bm) - 1) * q_stride_token + rp.q_ext;
  const int64_t o_span = (int64_t(bm) - 1) * out_stride_token + rp.o_ext;
  if (q_span > 0x3fffffff || o_span > 0x3fffffff)
    return mi::fail(MI_ERR_INVALID, "prefill run: q / out strides span %lld / %lld elements per tile (at most 2^30)",
                    (long long)q_span, (long long)o_span);
  const float scale = sm_scale > 0.f ? sm_scale : 1.0f / sqrtf(float(head_dim));
  rp.scale_log2 = scale * mi::kLog2e;
  const dim3 g{static_cast<uint32_t>(grid), 1u, 1u};
  switch (head_dim) {
    case 64: hipLaunchKernelGGL((prefill_run_kernel<64, 2>), g, dim3(64 * waves_for(64)), 0, s, rp); break;
    case 128: hipLaunchKernelGGL((prefill_run_kernel<128, 3>), g, dim3(64 * waves_for(128)), 0, s, rp); break;
    default: hipLaunchKernelGGL((prefill_run_kernel<256, 1>), g, dim3(64 * waves_for(256)), 0, s, rp); break;
  }
  return mi::check_launch("prefill_run_kernel");
}
