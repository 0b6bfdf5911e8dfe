// Stable expert-major routing on the device.
//
// Reference algorithm: runtime/routing.py:621-768 keeps routes whose expert
// id lies in [0, E), stable-argsorts them by expert id, and derives per-expert
// counts and exclusive offsets; kernels/fused_forward.py:158-480 builds the
// same order without a sort (private per-core histograms, an expert-major /
// core-minor prefix, then an order-preserving scatter) and
// kernels/fc2_combine.py:508-529 inverts it (route_to_send, -1 for drops).
//
// MI355X design: no global atomics, no host sync, no sort.
// Up to 1024 experts (route_fused_kernel): a unit is 2048 consecutive routes
// and one 16-wavefront workgroup. A workgroup needs, per expert, the routes in
// earlier units and in all units; up to 32768 routes it counts them itself from
// the ids (L2-resident), so routing is ONE launch; above, a first launch writes
// unit_counts[unit][expert], and every workgroup sums the table or a second
// launch scans it (see units_source). A block scan over the experts then
// gives every expert's
// first row, and each wavefront scatters its own 128 routes in order: a
// route's rank among equal experts comes from ballot match masks, the running
// counter per (wavefront, expert) sits in LDS, so the scatter is
// stable and needs no workgroup barrier. The last workgroup also writes the
// M-tile lists of the row GEMMs.
// It is latency-bound. Three launches (count, scan, scatter) without tile
// lists measured, against this form with them (graph replay, us): 8 routes
// over 128 experts 10.3 -> 6.4, 4084 over 60 17.6 -> 8.7, 32768 over 32 19.4
// -> 11.0, 65536 over 896 27.1 -> 17.7; each tile list built by itself was
// another 3 to 7 us launch, two per forward and two per backward.
// Above 1024 experts (up to 32768, bounded by LDS) count, scan and a
// one-wavefront scatter per unit remain three launches (the reference's
// lower-bound path for large bin counts, runtime/routing.py:246-416, serves
// the same range).
#include <mutex>

#include "common.h"

namespace {

constexpr int kThreads = 256;
constexpr int kChunk = 2048;                    // routes per unit
constexpr int kFusedThreads = 1024;
constexpr int kFusedWaves = kFusedThreads / 64;
constexpr int kSeg = kChunk / kFusedWaves;      // consecutive routes per wavefront of a unit
constexpr int kFusedExperts = 1024;             // LDS bound of route_fused_kernel (72 KiB)
constexpr int kMaxExperts = 32768;              // LDS bound of the 1-wave scatter (128 KiB) and the scan

__device__ __forceinline__ bool route_valid(int e, int E) { return e >= 0 && e < E; }

__global__ __launch_bounds__(kThreads) void route_count_kernel(const int32_t* __restrict__ sel,
                                                               int64_t R, int E, int nunits,
                                                               int32_t* __restrict__ unit_counts) {
  extern __shared__ int hist[];
  const int u = blockIdx.x;
  for (int e = threadIdx.x; e < E; e += kThreads) hist[e] = 0;
  __syncthreads();
  const int64_t start = static_cast<int64_t>(u) * kChunk;
  const int64_t end = min(R, start + kChunk);
  for (int64_t i = start + threadIdx.x; i < end; i += kThreads) {
    int e = sel[i];
    if (route_valid(e, E)) atomicAdd(&hist[e], 1);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += kThreads) unit_counts[static_cast<int64_t>(u) * E + e] = hist[e];
}

// Single workgroup: per-expert prefix over units, then an exclusive scan over
// experts. unit_counts[u][e] becomes the absolute first row of (u, e).
__global__ __launch_bounds__(1024) void route_scan_kernel(int32_t* __restrict__ unit_counts, int E,
                                                          int nunits, int32_t* __restrict__ counts,
                                                          int32_t* __restrict__ offsets) {
  extern __shared__ int tot[];  // E + 1024 scratch
  int* part = tot + E;
  const int tid = threadIdx.x;
  for (int e = tid; e < E; e += 1024) {
    int run = 0;
    int u = 0;
    for (; u + 8 <= nunits; u += 8) {
      int c[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) c[j] = unit_counts[static_cast<int64_t>(u + j) * E + e];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        unit_counts[static_cast<int64_t>(u + j) * E + e] = run;
        run += c[j];
      }
    }
    for (; u < nunits; ++u) {
      int c = unit_counts[static_cast<int64_t>(u) * E + e];
      unit_counts[static_cast<int64_t>(u) * E + e] = run;
      run += c;
    }
    tot[e] = run;
    counts[e] = run;
  }
  __syncthreads();
  // Exclusive scan of tot[0..E): each thread owns a contiguous slice.
  const int per = (E + 1023) / 1024;
  const int lo = min(E, tid * per), hi = min(E, lo + per);
  int s = 0;
  for (int e = lo; e < hi; ++e) s += tot[e];
  part[tid] = s;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {
    int v = tid >= off ? part[tid - off] : 0;
    __syncthreads();
    part[tid] += v;
    __syncthreads();
  }
  int base = part[tid] - s;
  for (int e = lo; e < hi; ++e) {
    int c = tot[e];
    tot[e] = base;
    offsets[e] = base;
    base += c;
  }
  if (tid == 1023) offsets[E] = part[1023];
  __syncthreads();
  for (int e = tid; e < E; e += 1024) {
    const int b = tot[e];
    for (int u = 0; u < nunits; ++u) unit_counts[static_cast<int64_t>(u) * E + e] += b;
  }
}

// Inclusive scan of v over the 1024 threads of a workgroup (wave shuffles,
// then the 16 wave totals); part is LDS scratch of kFusedWaves entries.
__device__ __forceinline__ uint64_t block_scan(uint64_t v, uint64_t* part) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint64_t o = __shfl_up(v, off);
    if (lane >= off) v += o;
  }
  if (lane == 63) part[wave] = v;
  __syncthreads();
  uint64_t base = 0;
#pragma unroll
  for (int w = 0; w < kFusedWaves; ++w) base += w < wave ? part[w] : 0;
  __syncthreads();
  return v + base;
}

// Where a unit's workgroup gets the routes of the other units from: it counts
// them itself, it sums the [nunits][E] table of route_count_kernel, or
// route_scan_kernel has turned that table into the unit's first rows.
enum { UNITS_RECOUNT = 0, UNITS_TABLE = 1, UNITS_SCANNED = 2 };

// One workgroup per unit, E <= kFusedExperts.
__global__ __launch_bounds__(kFusedThreads) void route_fused_kernel(
    const int32_t* __restrict__ sel, int64_t R, int top_k, int E, int nbits, int nunits, int source,
    const int32_t* __restrict__ unit_counts, const float* __restrict__ rw, int32_t* counts, int32_t* offsets,
    int32_t* __restrict__ send_route, int32_t* __restrict__ send_token,
    int32_t* __restrict__ route_to_send, float* __restrict__ weight_perm, TileList* __restrict__ tlS,
    TileList* __restrict__ tl256) {
  // [wave][expert]: routes of the segment, then its next row
  __shared__ __attribute__((aligned(16))) int seg[kFusedWaves * kFusedExperts];
  __shared__ int before[kFusedExperts], rest[kFusedExperts];  // routes in earlier / later units
  __shared__ uint64_t part[kFusedWaves];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int u = blockIdx.x;
  const int64_t start = static_cast<int64_t>(u) * kChunk;
  const int64_t end = min(R, start + kChunk);
  for (int i = tid; i < kFusedWaves * E; i += kFusedThreads) seg[i] = 0;
  for (int e = tid; e < E; e += kFusedThreads) before[e] = rest[e] = 0;
  __syncthreads();

  // own unit: wave w owns routes start + w * kSeg ..
  constexpr int ITERS = kSeg / 64;
  int key[ITERS];
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int64_t i = start + wave * kSeg + it * 64 + lane;
    const int e = i < R ? sel[i] : -1;
    key[it] = route_valid(e, E) ? e : E;
  }
  if (source == UNITS_SCANNED) {
    for (int e = tid; e < E; e += kFusedThreads) before[e] = unit_counts[static_cast<int64_t>(u) * E + e];
  } else if (source == UNITS_TABLE) {
    // thread (g, e) sums column e of every G-th row, 16 rows in flight
    const int G = kFusedThreads / E, g = tid / E, e = tid - g * E;
    if (g < G) {
      int b = 0, r = 0;
      for (int v = g; v < nunits; v += 16 * G) {
        int c[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) c[j] = unit_counts[static_cast<int64_t>(min(v + j * G, nunits - 1)) * E + e];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int w = v + j * G;
          b += w < u ? c[j] : 0;
          r += w > u && w < nunits ? c[j] : 0;
        }
      }
      atomicAdd(&before[e], b);
      atomicAdd(&rest[e], r);
    }
  } else if (nunits > 1) {
    // Eight copies of each histogram (in seg, not yet in use), one per eight
    // lanes: ids that repeat within a wavefront (a hot expert's) queue up on
    // their LDS word.
    const int copy = (lane >> 3) & 7;
    auto count = [&](int64_t lo, int64_t hi, int* hist) {
      int64_t i = lo + tid;
      for (; i + 7 * kFusedThreads < hi; i += 8 * kFusedThreads) {
        int e[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) e[j] = sel[i + j * kFusedThreads];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (route_valid(e[j], E)) atomicAdd(&hist[e[j] * 8 + copy], 1);
      }
      for (; i < hi; i += kFusedThreads) {
        const int e = sel[i];
        if (route_valid(e, E)) atomicAdd(&hist[e * 8 + copy], 1);
      }
    };
    static_assert(kFusedWaves == 16, "two histograms of eight copies fill seg");
    count(0, start, seg);
    count(end, R, seg + 8 * E);
    __syncthreads();
    if (tid < E) {
      auto take = [](int* p) {  // sums a copy set and clears it
        int4* q = reinterpret_cast<int4*>(p);
        const int4 a = q[0], b = q[1];
        q[0] = q[1] = make_int4(0, 0, 0, 0);
        return a.x + a.y + a.z + a.w + b.x + b.y + b.z + b.w;
      };
      before[tid] = take(seg + tid * 8);
      rest[tid] = take(seg + (E + tid) * 8);
    }
    __syncthreads();
  }
#pragma unroll
  for (int it = 0; it < ITERS; ++it)
    if (key[it] < E) atomicAdd(&seg[wave * E + key[it]], 1);
  __syncthreads();

  // per expert: first row of every segment relative to the expert, then the
  // expert's first row from a scan over the experts
  int total = 0;
  if (tid < E) {
    int run = before[tid];
#pragma unroll
    for (int w = 0; w < kFusedWaves; ++w) {
      const int c = seg[w * E + tid];
      seg[w * E + tid] = run;
      run += c;
    }
    total = run + rest[tid];
  }
  int first = 0;
  if (source == UNITS_SCANNED) {  // the rows are absolute, counts and offsets written
    if (tid < E) {
      first = offsets[tid];
      total = counts[tid];
    }
  } else {
    first = static_cast<int>(block_scan(static_cast<uint64_t>(total), part)) - total;
  }
  if (tid < E && source != UNITS_SCANNED) {
#pragma unroll
    for (int w = 0; w < kFusedWaves; ++w) seg[w * E + tid] += first;
    if (u == 0) {
      counts[tid] = total;
      offsets[tid] = first;
      if (tid == E - 1) offsets[E] = first + total;
    }
  }
  if (u == nunits - 1 && tlS) {
    const uint64_t tS = (total + kStreamRows - 1) / kStreamRows, t256 = (total + 255) / 256;
    const uint64_t t = block_scan(tS | (t256 << 32), part);
    if (tid < E) {
      int n = static_cast<int>(t & 0xffffffffu) - static_cast<int>(tS);
      for (int r = 0; r < total; r += kStreamRows)
        tlS->tiles[n++] = make_int4(tid, first + r, first + min(r + kStreamRows, total), 0);
      n = static_cast<int>(t >> 32) - static_cast<int>(t256);
      for (int r = 0; r < total; r += 256) tl256->tiles[n++] = make_int4(tid, first + r, first + min(r + 256, total), 0);
    }
    if (tid == kFusedThreads - 1) {
      tlS->count = static_cast<int>(t & 0xffffffffu);
      tl256->count = static_cast<int>(t >> 32);
    }
  }
  __syncthreads();

  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  int* next = seg + wave * E;  // this wavefront's counters: LDS operations of one wave stay in order
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int64_t i = start + wave * kSeg + it * 64 + lane;
    const bool present = i < R, valid = key[it] < E;
    uint64_t mask = __ballot(1);  // lanes holding the same key
    for (int b = 0; b < nbits; ++b) {
      const bool bit = (key[it] >> b) & 1;
      const uint64_t m = __ballot(bit);
      mask &= bit ? m : ~m;
    }
    const int rank = __popcll(mask & lt_mask);
    const int base = valid ? next[key[it]] : 0;
    asm volatile("" ::: "memory");  // every lane reads its counter before a leader moves it
    if (valid && rank == 0) next[key[it]] = base + __popcll(mask);
    asm volatile("" ::: "memory");
    if (present) {
      const int pos = valid ? base + rank : -1;
      route_to_send[i] = pos;
      if (valid) {
        send_route[pos] = static_cast<int32_t>(i);
        send_token[pos] = static_cast<int32_t>(i / top_k);
        if (weight_perm != nullptr) weight_perm[pos] = rw[i];
      }
    }
  }
}

// Scatter for large expert counts (E > kFusedExperts): one wavefront per unit,
// so the stable rank of a route among equal experts comes from the ballot
// match mask alone and LDS holds only the E running row counters.
__global__ __launch_bounds__(64) void route_scatter_wave_kernel(
    const int32_t* __restrict__ sel, int64_t R, int top_k, int E, int nbits,
    const int32_t* __restrict__ unit_base, const float* __restrict__ rw,
    int32_t* __restrict__ send_route, int32_t* __restrict__ send_token,
    int32_t* __restrict__ route_to_send, float* __restrict__ weight_perm) {
  extern __shared__ int run[];  // [E] next free row of each expert
  const int u = blockIdx.x;
  const int lane = threadIdx.x;
  for (int e = lane; e < E; e += 64) run[e] = unit_base[static_cast<int64_t>(u) * E + e];
  __syncthreads();
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  const int64_t start = static_cast<int64_t>(u) * kChunk;
  for (int it = 0; it < kChunk / 64; ++it) {
    const int64_t i = start + static_cast<int64_t>(it) * 64 + lane;
    const bool present = i < R;
    const int e = present ? sel[i] : -1;
    const bool valid = present && route_valid(e, E);
    const int key = valid ? e : E;
    uint64_t mask = __ballot(1);
    for (int b = 0; b < nbits; ++b) {
      const bool bit = (key >> b) & 1;
      const uint64_t m = __ballot(bit);
      mask &= bit ? m : ~m;
    }
    const int rank = __popcll(mask & lt_mask);
    const int base = valid ? run[key] : 0;
    __syncthreads();  // every lane has read its expert's counter
    if (present) {
      if (valid) {
        const int pos = base + rank;
        send_route[pos] = static_cast<int32_t>(i);
        send_token[pos] = static_cast<int32_t>(i / top_k);
        route_to_send[i] = pos;
        if (weight_perm != nullptr) weight_perm[pos] = rw[i];
        if (rank == 0) run[key] = base + __popcll(mask);
      } else {
        route_to_send[i] = -1;
      }
    }
    __syncthreads();
  }
}

}  // namespace

extern "C" size_t mm_route_workspace_bytes(int64_t num_routes, int32_t num_experts) {
  const int64_t nunits = (num_routes + kChunk - 1) / kChunk;
  return mm_align_up(static_cast<size_t>(nunits) * static_cast<size_t>(num_experts) * 4 + 256, 256);
}

namespace {

// Recounting costs each workgroup R ids and their LDS atomics, the table its
// R / 2048 * E entries and a launch. Measured (us, recount / table): 32768
// routes over 8 experts 10.6 / 11.6, over 896 13.3 / 14.5; 65536 over 8 14.2 /
// 9.8, over 896 16.1 / 16.3. With every id the same the atomics of a histogram
// queue up: 32768 routes 13.9 / 11.6 with the eight copies (one histogram: 33;
// 524288 over 896 experts: 450, the table 36).
// Reading the table grows with the square of R, the scan does not: it takes
// over at 6e8 entries over all units (summed / scanned: 1048576 routes over
// 1024 experts, 2.7e8, 134 / 159; 4194304 over 128, 5.4e8, 246 / 377; over
// 512, 2.1e9, 790 / 507).
int units_source(int64_t num_routes, int E, int64_t nunits) {
  if (num_routes <= 32768) return UNITS_RECOUNT;
  return nunits * nunits * E > 600000000 ? UNITS_SCANNED : UNITS_TABLE;
}

int route_launch(const int32_t* selected, int64_t num_routes, int32_t top_k, int32_t num_experts,
                 const float* routing_weights, int32_t* counts, int32_t* offsets, int32_t* send_route,
                 int32_t* send_token, int32_t* route_to_send, float* weight_perm, int32_t* unit_counts,
                 void* tiles, hipStream_t s, const char* what) {
  const int E = num_experts;
  const int nunits = static_cast<int>((num_routes + kChunk - 1) / kChunk);
  const int nbits = 32 - __builtin_clz(static_cast<unsigned>(E));
  TileList* tlS = tiles ? mm_tile_list_of(tiles, num_routes, E, kStreamRows) : nullptr;
  TileList* tl256 = tiles ? mm_tile_list_of(tiles, num_routes, E, 256) : nullptr;
  if (E <= kFusedExperts) {
    const int source = units_source(num_routes, E, nunits);
    if (source != UNITS_RECOUNT)
      route_count_kernel<<<nunits, kThreads, E * sizeof(int), s>>>(selected, num_routes, E, nunits, unit_counts);
    if (source == UNITS_SCANNED)
      route_scan_kernel<<<1, 1024, (E + 1024) * sizeof(int), s>>>(unit_counts, E, nunits, counts, offsets);
    route_fused_kernel<<<nunits > 0 ? nunits : 1, kFusedThreads, 0, s>>>(
        selected, num_routes, top_k, E, nbits, nunits > 0 ? nunits : 1, source,
        unit_counts, routing_weights, counts, offsets, send_route, send_token, route_to_send, weight_perm, tlS, tl256);
    return mm_check_launch(what);
  }
  // dynamic LDS above 64 KiB (up to 132 KiB at kMaxExperts); set once
  static std::once_flag once;
  std::call_once(once, [] {
    const int bytes = (kMaxExperts + 1024) * static_cast<int>(sizeof(int));
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(route_count_kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(route_scan_kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(route_scatter_wave_kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  });
  if (nunits > 0)
    route_count_kernel<<<nunits, kThreads, E * sizeof(int), s>>>(selected, num_routes, E, nunits, unit_counts);
  route_scan_kernel<<<1, 1024, (E + 1024) * sizeof(int), s>>>(unit_counts, E, nunits, counts, offsets);
  if (nunits > 0)
    route_scatter_wave_kernel<<<nunits, 64, static_cast<size_t>(E) * sizeof(int), s>>>(
        selected, num_routes, top_k, E, nbits, unit_counts, routing_weights, send_route, send_token,
        route_to_send, weight_perm);
  if (int rc = mm_check_launch(what)) return rc;
  if (tiles) {
    if (int rc = mm_build_tiles(offsets, E, kStreamRows, tlS, s)) return rc;
    return mm_build_tiles(offsets, E, 256, tl256, s);
  }
  return MM_OK;
}

}  // namespace

#define MM_ROUTE_CHECK_ARGS(what)                                                                          \
  MM_CHECK_ARG(num_routes >= 0 && num_routes < (int64_t(1) << 31), what ": num_routes out of range");     \
  MM_CHECK_ARG(top_k > 0, what ": top_k must be positive");                                                \
  MM_CHECK_ARG(num_experts > 0 && num_experts <= kMaxExperts, what ": num_experts must be in [1, %d]",     \
               kMaxExperts);                                                                               \
  MM_CHECK_ARG(counts && offsets, what ": counts/offsets must be non-null");                               \
  MM_CHECK_ARG(num_routes == 0 || (selected && send_route && send_token && route_to_send),                 \
               what ": route tables must be non-null");                                                    \
  MM_CHECK_ARG((weight_perm == nullptr) == (routing_weights == nullptr),                                   \
               what ": routing_weights and weight_perm must be given together")

extern "C" int mm_route(const int32_t* selected, int64_t num_routes, int32_t top_k, int32_t num_experts,
                        const float* routing_weights, int32_t* counts, int32_t* offsets,
                        int32_t* send_route, int32_t* send_token, int32_t* route_to_send,
                        float* weight_perm, void* workspace, size_t workspace_bytes,
                        mm_stream_t stream) {
  MM_ROUTE_CHECK_ARGS("mm_route");
  if (workspace_bytes < mm_route_workspace_bytes(num_routes, num_experts) || workspace == nullptr) {
    mm_set_error("mm_route: workspace too small");
    return MM_E_WS;
  }
  return route_launch(selected, num_routes, top_k, num_experts, routing_weights, counts, offsets, send_route,
                      send_token, route_to_send, weight_perm, static_cast<int32_t*>(workspace), nullptr,
                      mm_hip_stream(stream), "mm_route");
}

extern "C" size_t mm_tile_lists_size(int64_t max_rows, int32_t num_experts) {
  return mm_tile_lists_bytes(max_rows, num_experts);
}

extern "C" int mm_route_tiles(const int32_t* selected, int64_t num_routes, int32_t top_k, int32_t num_experts,
                              const float* routing_weights, int32_t* counts, int32_t* offsets,
                              int32_t* send_route, int32_t* send_token, int32_t* route_to_send,
                              float* weight_perm, void* tiles, size_t tiles_bytes, void* workspace,
                              size_t workspace_bytes, mm_stream_t stream) {
  MM_ROUTE_CHECK_ARGS("mm_route_tiles");
  if (workspace_bytes < mm_route_workspace_bytes(num_routes, num_experts) || workspace == nullptr) {
    mm_set_error("mm_route_tiles: workspace too small");
    return MM_E_WS;
  }
  if (tiles == nullptr || (reinterpret_cast<uintptr_t>(tiles) & 15u) ||
      tiles_bytes < mm_tile_lists_bytes(num_routes, num_experts)) {
    mm_set_error("mm_route_tiles: tile lists need %zu bytes, 16-byte aligned",
                 mm_tile_lists_bytes(num_routes, num_experts));
    return MM_E_WS;
  }
  return route_launch(selected, num_routes, top_k, num_experts, routing_weights, counts, offsets, send_route,
                      send_token, route_to_send, weight_perm, static_cast<int32_t*>(workspace), tiles,
                      mm_hip_stream(stream), "mm_route_tiles");
}

// ---------------------------------------------------------------- no-allocation variant
//
// mm_route_noalloc keeps the per-unit count table (the only scratch mm_route
// uses) in a file-scope device array instead of a caller workspace. Every
// GPU the library runs on holds its own copy until the process ends; the
// host reaches it through the address hipGetSymbolAddress returns on that
// device (the array's name in host code is only a stand-in). The table is
// fully rewritten by route_count_kernel on every call, so nothing needs
// clearing; calls that overlap on one GPU (different streams) race on it.
namespace {

constexpr size_t kRouteScratchBytes = size_t(4) << 20;  // 4 MiB
static __device__ __align__(256) int32_t scratch[kRouteScratchBytes / sizeof(int32_t)];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
int32_t* g_scratch_ptr[kMaxDevices] = {nullptr};

int scratch_for_current_device(int32_t** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    mm_set_error("mm_route_noalloc: no usable current device (%s)", hipGetErrorString(e));
    return MM_E_LAUNCH;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
      mm_set_error("mm_route_noalloc: hipGetSymbolAddress failed (%s)", hipGetErrorString(e));
      return MM_E_LAUNCH;
    }
    g_scratch_ptr[dev] = static_cast<int32_t*>(p);
  }
  *out = g_scratch_ptr[dev];
  return MM_OK;
}

}  // namespace

extern "C" size_t mm_route_noalloc_scratch_bytes(void) { return kRouteScratchBytes; }

extern "C" int mm_route_noalloc(const int32_t* selected, int64_t num_routes, int32_t top_k,
                                int32_t num_experts, const float* routing_weights, int32_t* counts,
                                int32_t* offsets, int32_t* send_route, int32_t* send_token,
                                int32_t* route_to_send, float* weight_perm, mm_stream_t stream) {
  MM_ROUTE_CHECK_ARGS("mm_route_noalloc");
  const size_t need = mm_route_workspace_bytes(num_routes, num_experts);
  if (need > kRouteScratchBytes) {
    mm_set_error("mm_route_noalloc: %lld routes x %d experts need %zu bytes of scratch, above the %zu-byte "
                 "maximum; use mm_route with a workspace",
                 static_cast<long long>(num_routes), num_experts, need, kRouteScratchBytes);
    return MM_E_ARG;
  }
  int32_t* ws = nullptr;
  if (int rc = scratch_for_current_device(&ws)) return rc;
  return route_launch(selected, num_routes, top_k, num_experts, routing_weights, counts, offsets, send_route,
                      send_token, route_to_send, weight_perm, ws, nullptr, mm_hip_stream(stream), "mm_route_noalloc");
}
