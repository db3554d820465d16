// SPDX-License-Identifier: Apache-2.0
//
// The routes of one local expert, found by the workgroup that serves it (decode products without
// a sort): the routes whose id is the expert's, in route order - the order the sort's stable
// placement gives them.
#pragma once

#include "common.hpp"

namespace uniserve {

/// The most routes an expert-major workgroup lists (a decode batch's).
constexpr int kExpertRoutes = 4096;

/// Routes each wavefront of a kWaves-wave workgroup scans (whole chunks of 64).
template <int kWaves>
__host__ __device__ constexpr int64_t routes_per_wave(int64_t routes) {
  return ((routes + kWave - 1) / kWave + kWaves - 1) / kWaves * kWave;
}

/// A wavefront's first 4 x 64 route ids of its stretch (as list_expert_routes scans it), loaded
/// ahead: a kernel that issues its first weight loads between these loads and the scan waits for
/// the ids alone (the wait for a load also waits for every load issued before it).
struct FirstRouteIds {
  int32_t id[4];
};
template <int kWaves>
__device__ __forceinline__ FirstRouteIds load_first_route_ids(const int32_t *ids, int64_t routes) {
  const int wave = static_cast<int>(threadIdx.x) / kWave;
  const int64_t begin = wave * routes_per_wave<kWaves>(routes);
  FirstRouteIds first;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int64_t route = begin + u * kWave + lane_id();
    first.id[u] = ids[route < routes ? route : 0];  // (the scan drops routes past its stretch)
  }
  return first;
}

/// Lists the live routes (route < live) whose id is `want`: wavefront w ballots routes
/// [w q, (w + 1) q), q = routes_per_wave, into list[w q ..] and counts[w]; counts[kWaves] is the
/// total. Every thread of the workgroup calls it (two barriers); returns the total.
/// `first`, if given: load_first_route_ids' ids, used for the stretch's first 4 x 64 routes.
template <int kWaves>
__device__ __forceinline__ int list_expert_routes(const int32_t *ids, int64_t routes, int64_t live, int32_t want,
                                                  int32_t *list, int32_t *counts,
                                                  const FirstRouteIds *first = nullptr) {
  const int wave = static_cast<int>(threadIdx.x) / kWave;
  const int lane = lane_id();
  const int64_t per_wave = routes_per_wave<kWaves>(routes);
  const int64_t begin = wave * per_wave;
  const int64_t end = begin + per_wave < routes ? begin + per_wave : routes;
  int32_t *mine = list + wave * per_wave;
  int count = 0;
  for (int64_t c = begin; c < end; c += 4 * kWave) {
    int32_t id[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t route = c + u * kWave + lane;
      const bool held = route < end && route < live;
      if (first != nullptr && c == begin) id[u] = held ? first->id[u] : -1;
      else id[u] = held ? ids[route] : -1;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool match = id[u] == want;
      const uint64_t mask = __ballot(match);
      if (match) mine[count + __popcll(mask & ((1ull << lane) - 1))] = static_cast<int32_t>(c + u * kWave + lane);
      count += __popcll(mask);
    }
  }
  if (lane == 0) counts[wave] = count;
  __syncthreads();
  if (threadIdx.x == 0) {
    int total = 0;
    for (int w = 0; w < kWaves; ++w) total += counts[w];
    counts[kWaves] = total;
  }
  __syncthreads();
  return counts[kWaves];
}

/// Local experts a compact grid can tell apart (the fused front end's window bound).
constexpr int kPresentExperts = 512;

/// The n-th smallest local expert that some live route names, or -1 when fewer are named: the
/// workgroup marks the named experts in an LDS bitmap (`bits`, kPresentExperts / 32 words) and
/// every thread counts its way to the n-th mark. Every thread of the workgroup calls it (two
/// barriers) and gets the same answer.
template <int kThreads>
__device__ __forceinline__ int32_t nth_named_expert(const int32_t *ids, int64_t routes, int64_t live, int32_t local_offset,
                                                    int32_t local_experts, int n, uint32_t *bits) {
  constexpr int kWords = kPresentExperts / 32;
  if (threadIdx.x < kWords) bits[threadIdx.x] = 0u;
  __syncthreads();
  const int64_t last = routes < live ? routes : live;
  for (int64_t route = threadIdx.x; route < last; route += kThreads) {
    const int32_t local = ids[route] - local_offset;
    if (local >= 0 && local < local_experts) atomicOr(bits + local / 32, 1u << (local % 32));
  }
  __syncthreads();
  for (int w = 0; w < kWords; ++w) {
    uint32_t word = bits[w];
    const int count = __popc(word);
    if (n >= count) {
      n -= count;
      continue;
    }
    for (; n > 0; --n) word &= word - 1;  // drop the n lowest marks
    return 32 * w + __ffs(static_cast<int>(word)) - 1;
  }
  return -1;
}

/// A run of an expert's listed rows.
struct RowRun {
  int32_t expert;  ///< local expert, or -1: no such run
  int32_t first;   ///< its first row
  int32_t rows;    ///< rows it covers (the expert's last run: fewer may be left)
};

/// The n-th of at most `columns` runs (columns >= the smaller of local_experts and
/// (routes - 1) / kRows) covering every row past the experts' first kRows each, experts ascending,
/// rows ascending: runs of kRows rows, or of the smallest doubling of it with which `columns` runs
/// are enough. The workgroup counts every local expert's live routes in `counts` (LDS,
/// local_experts words) and scans the experts' run counts. Every thread of the workgroup calls it
/// and gets the same answer; `counts` is free again when it returns.
template <int kThreads, int kRows>
__device__ __forceinline__ RowRun nth_extra_run(const int32_t *ids, int64_t routes, int64_t live, int32_t local_offset,
                                                int32_t local_experts, int n, int columns, int32_t *counts) {
  constexpr int kWaves = kThreads / kWave;
  __shared__ int32_t wave_runs[2][kWaves];
  __shared__ RowRun found;
  const int t = static_cast<int>(threadIdx.x);
  for (int e = t; e < local_experts; e += kThreads) counts[e] = 0;
  if (t == 0) found = RowRun{-1, 0, 0};
  __syncthreads();
  const int64_t last = routes < live ? routes : live;
  constexpr int kAhead = 8;  // ids in flight per thread
  for (int64_t at = t; at < last; at += kAhead * kThreads) {
    int32_t local[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int64_t route = at + u * kThreads;
      local[u] = route < last ? ids[route] - local_offset : -1;
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      if (local[u] >= 0 && local[u] < local_experts) atomicAdd(counts + local[u], 1);
  }
  __syncthreads();
  // Thread t's experts: [t each, (t + 1) each).
  const int each = (local_experts + kThreads - 1) / kThreads;
  auto runs_of = [&](int e, int rows) { return e < local_experts && counts[e] > kRows ? (counts[e] - kRows + rows - 1) / rows : 0; };
  int rows = kRows, own, upto, parity = 0;
  for (;; rows *= 2, parity ^= 1) {
    own = 0;
    for (int i = 0; i < each; ++i) own += runs_of(t * each + i, rows);
    upto = own;  // inclusive scan over the wavefront
#pragma unroll
    for (int step = 1; step < kWave; step *= 2) {
      const int before = __shfl_up(upto, step, kWave);
      if (lane_id() >= step) upto += before;
    }
    if (lane_id() == kWave - 1) wave_runs[parity][t / kWave] = upto;
    __syncthreads();
    int total = 0;
    for (int w = 0; w < kWaves; ++w) total += wave_runs[parity][w];
    if (total <= columns || rows >= static_cast<int>(routes)) break;  // (uniform; one run per expert at most)
  }
  int at = upto - own;
  for (int w = 0; w < t / kWave; ++w) at += wave_runs[parity][w];
  if (n >= at && n < at + own) {
    for (int i = 0; i < each; ++i) {
      const int runs = runs_of(t * each + i, rows);
      if (n < at + runs) {
        found = RowRun{t * each + i, kRows + (n - at) * rows, rows};
        break;
      }
      at += runs;
    }
  }
  __syncthreads();
  return found;
}

/// What one workgroup of a wide kernel (a one-dimensional grid of (columns + extra_columns) * slices)
/// serves: rows [row_first, row_last) of `expert`'s, its `slice`-th run of weight rows.
struct ColumnWork {
  int32_t expert;  ///< local expert, or -1: nothing
  int32_t slice;
  int32_t row_first, row_last;
};

/// The first columns * slices workgroups serve a column - an expert, or with `compact` the n-th named
/// one - each, slice by slice, and the last extra_columns * slices the rows past an expert's first
/// kPassRows, where any has more (nth_extra_run), run by run, so that the runs there are start first and
/// the workgroups that find none come last (slice by slice: 235B e4m3, window of 32 experts, Zipf, T=383
/// 514 us against 362, 30B bf16, every expert, Zipf, T=301 255 against 238). Every thread of the workgroup calls it; `list` holds
/// local_experts words and is free again when it returns.
template <int kThreads, int kPassRows, class Params>
__device__ __forceinline__ ColumnWork column_work(const Params &p, int64_t live, int slices, int32_t *list) {
  __shared__ uint32_t named[kPresentExperts / 32];
  ColumnWork work{-1, 0, 0, 0x7fffffff};
  const int b = static_cast<int>(blockIdx.x);
  const int own = p.columns * slices;
  const bool is_extra = b >= own;
  work.slice = is_extra ? (b - own) % slices : b / p.columns;
  const int column = is_extra ? (b - own) / slices : b - work.slice * p.columns;
  const int32_t offset = static_cast<int32_t>(p.local_offset), experts = static_cast<int32_t>(p.local_experts);
  if (is_extra) {
    const RowRun run = nth_extra_run<kThreads, kPassRows>(p.ids, p.routes, live, offset, experts, column, p.extra_columns, list);
    work.expert = run.expert;
    work.row_first = run.first;
    work.row_last = run.first + run.rows;
    return work;
  }
  work.expert = p.compact ? nth_named_expert<kThreads>(p.ids, p.routes, live, offset, experts, column, named) : column;
  if (p.extra_columns > 0) work.row_last = kPassRows;
  return work;
}

/// A window of few much-named experts needs more runs than it has experts, and a near-uniform one pays
/// for the workgroups that find none. Layer, sixteen 235B experts from the first, Zipf / near-uniform:
/// e4m3 T=383 with 16 columns 516 / 98 us, with 48 320 / 101, with all of 95 292 / 110; 30B bf16 T=300 237
/// / 52, 151 / 56, 138 / 58.
constexpr int64_t kMostExtraColumns = 48;

/// The extra columns a launch needs: one per run of `pass_rows` that may lie past an expert's first
/// (never more than the experts, or kMostExtraColumns if the experts are fewer), none for a compact
/// grid or where no expert is likely to have more than two passes of rows (`tokens`, unless the slot map
/// names a slot twice).
inline int32_t extra_columns(int64_t routes, int64_t top, int64_t local_experts, bool compact, int64_t pass_rows) {
  const int64_t runs = (routes - 1) / pass_rows;
  if (compact || routes <= 2 * pass_rows * top) return 0;
  const int64_t most = local_experts > kMostExtraColumns ? local_experts : kMostExtraColumns;
  return static_cast<int32_t>(runs < most ? runs : most);
}

/// Row m of the list (m < the total).
template <int kWaves>
__device__ __forceinline__ int64_t listed_route(const int32_t *list, const int32_t *counts, int64_t routes, int m) {
  int w = 0;
  int before = 0;
  while (w + 1 < kWaves && m >= before + counts[w]) before += counts[w++];
  return list[w * routes_per_wave<kWaves>(routes) + (m - before)];
}

}  // namespace uniserve
