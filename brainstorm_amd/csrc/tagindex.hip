// Tag-index gather: merging the rows that several paths produced for the same cell.
//
// The reference does this with library calls (src/backend/torch/router.cc): the per-path tag
// vectors are concatenated and passed to `_unique(sorted, return_inverse)` (:348-369), a sort;
// the inverse is then expanded to one int64 index per *element* (`repeat`, :451) and the rows are
// summed with `scatter_reduce` (:449-472), whose atomics add in no fixed order.
//
// Here neither step sorts or expands anything.
//   * unique: the tags lie in a known range [lo, hi]; a presence table over that range, one
//     prefix sum over it (which is the rank of every tag in the sorted unique list) and a lookup
//     per row give the unique tags and the inverse.
//   * sum: every row is pushed on a linked list of its output row with one atomic exchange; a
//     wavefront per output row walks its list (one hop per contributing path), orders the row
//     numbers in registers and adds the rows in ascending row order in fp32, so the result does
//     not depend on the order in which the atomics landed and every output row is written once.
#include <algorithm>
#include <climits>
#include <type_traits>

#include "common.hpp"
#include "rows.hpp"

namespace brt {
namespace {

constexpr int kScanThreads = 1024;
constexpr int kScanItems = 8;
constexpr int kScanChunk = kScanThreads * kScanItems;
constexpr long kMaxRange = 1l << 25;  // 4096 scan blocks; each block adds up the totals before it

__global__ void fill_zero_kernel(int* __restrict__ p, long n) {
  const long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

template <typename K>
__global__ void mark_present_kernel(const K* __restrict__ keys, long n, long lo, long range,
                                    int* __restrict__ present) {
  const long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const long k = static_cast<long>(keys[i]) - lo;
  if (k >= 0 && k < range) present[k] = 1;  // every writer stores the same value
}

// Sum of one block's chunk of the presence table.
__global__ __launch_bounds__(kScanThreads) void chunk_total_kernel(const int* __restrict__ present,
                                                                   long range, int* __restrict__ totals) {
  __shared__ int s_wave[kScanThreads / kWave];
  const long base = static_cast<long>(blockIdx.x) * kScanChunk + threadIdx.x * kScanItems;
  int v = 0;
#pragma unroll
  for (int i = 0; i < kScanItems; ++i)
    if (base + i < range) v += present[base + i];
  const int incl = wave_inclusive_scan(v);
  if (lane_id() == kWave - 1) s_wave[threadIdx.x >> 6] = incl;
  __syncthreads();
  if (threadIdx.x == 0) {
    int t = 0;
    for (int w = 0; w < kScanThreads / kWave; ++w) t += s_wave[w];
    totals[blockIdx.x] = t;
  }
}

// Turns the presence table into ranks (exclusive prefix sums, in place) and writes the present
// keys, in ascending order, to `unique`; the last block stores how many there are.
template <typename K>
__global__ __launch_bounds__(kScanThreads) void rank_emit_kernel(int* __restrict__ table, long range,
                                                                 const int* __restrict__ totals, long lo,
                                                                 K* __restrict__ unique,
                                                                 int* __restrict__ n_unique) {
  __shared__ int s_wave[kScanThreads / kWave];
  __shared__ int s_before;
  const int tid = threadIdx.x, wave = tid >> 6;
  // keys of the blocks before this one
  if (wave == 0) {
    int t = 0;
    for (int b = tid; b < static_cast<int>(blockIdx.x); b += kWave) t += totals[b];
    const int incl = wave_inclusive_scan(t);
    if (tid == kWave - 1) s_before = incl;
  }
  const long base = static_cast<long>(blockIdx.x) * kScanChunk + tid * kScanItems;
  int flag[kScanItems];
  int mine = 0;
#pragma unroll
  for (int i = 0; i < kScanItems; ++i) {
    flag[i] = base + i < range ? table[base + i] : 0;
    mine += flag[i];
  }
  const int incl = wave_inclusive_scan(mine);
  if (lane_id() == kWave - 1) s_wave[wave] = incl;
  __syncthreads();
  int rank = s_before + incl - mine;
  for (int w = 0; w < wave; ++w) rank += s_wave[w];
#pragma unroll
  for (int i = 0; i < kScanItems; ++i) {
    if (base + i < range) {
      table[base + i] = rank;
      if (flag[i]) unique[rank] = static_cast<K>(lo + base + i);
      rank += flag[i];
    }
  }
  if (blockIdx.x == gridDim.x - 1 && tid == kScanThreads - 1) *n_unique = rank;
}

template <typename K>
__global__ void inverse_kernel(const K* __restrict__ keys, long n, long lo, long range,
                               const int* __restrict__ rank, int64_t* __restrict__ inverse) {
  const long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const long k = static_cast<long>(keys[i]) - lo;
  inverse[i] = (k >= 0 && k < range) ? rank[k] : -1;
}

// The whole unique in one workgroup, the table in LDS: for ranges of up to kSmallRange tags and
// inputs short enough for 1024 threads to walk twice.
constexpr int kSmallRange = 32768;
constexpr long kSmallCount = BRT_UNIQUE_WHOLE_MAX;

constexpr int kKeysInFlight = 8;

// A batch of keys per thread.  The loads are unconditional (an index past the end reads the last key
// again and is dropped), all in flight together; one at a time, every key would be a memory round
// trip of its own for this one workgroup.
template <typename K>
__device__ __forceinline__ void key_batch(const K* __restrict__ keys, int n, int base, K (&v)[kKeysInFlight]) {
#pragma unroll
  for (int j = 0; j < kKeysInFlight; ++j)
    v[j] = keys[min(base + j * kScanThreads + static_cast<int>(threadIdx.x), n - 1)];  // n >= 1
}

// The rank of every tag in the table, and the unique tags.  The number of unique keys is returned to the last thread; the first
// batch of keys, `held`, is in registers.
template <typename K>
__device__ __forceinline__ int ranks_in_lds(const K* __restrict__ keys, int n, long lo, int range, const K (&held)[kKeysInFlight],
                                            K* __restrict__ unique, int* s_table) {
  __shared__ int s_wave[kScanThreads / kWave];
  const int tid = threadIdx.x, wave = tid >> 6;
  for (int i = tid; i < range; i += kScanThreads) s_table[i] = 0;
  __syncthreads();
  for (int base = 0; base < n; base += kKeysInFlight * kScanThreads) {
    K v[kKeysInFlight];
    if (base == 0) {
#pragma unroll
      for (int j = 0; j < kKeysInFlight; ++j) v[j] = held[j];
    } else {
      key_batch(keys, n, base, v);
    }
#pragma unroll
    for (int j = 0; j < kKeysInFlight; ++j) {
      const long k = static_cast<long>(v[j]) - lo;
      if (base + j * kScanThreads + tid < n && k >= 0 && k < range) s_table[k] = 1;
    }
  }
  __syncthreads();
  // every thread scans a run of consecutive entries; an odd run length keeps the lanes of a
  // wavefront on different LDS banks
  const int run = ((range + kScanThreads - 1) / kScanThreads) | 1;
  const int first = min(tid * run, range), last = min(first + run, range);
  int mine = 0;
  for (int i = first; i < last; ++i) mine += s_table[i];
  const int incl = wave_inclusive_scan(mine);
  if (lane_id() == kWave - 1) s_wave[wave] = incl;
  __syncthreads();
  int rank = incl - mine;
  for (int w = 0; w < wave; ++w) rank += s_wave[w];
  for (int i = first; i < last; ++i) {
    const int flag = s_table[i];
    s_table[i] = rank;
    if (flag) unique[rank] = static_cast<K>(lo + i);
    rank += flag;
  }
  __syncthreads();
  return rank;
}

// ... and the inverse, for which the first batch of keys stays in registers.
template <typename K>
__device__ __forceinline__ int unique_in_lds(const K* __restrict__ keys, int n, long lo, int range, const K (&held)[kKeysInFlight],
                                             K* __restrict__ unique, int64_t* __restrict__ inverse, int* s_table) {
  const int tid = threadIdx.x;
  const int rank = ranks_in_lds(keys, n, lo, range, held, unique, s_table);
  for (int base = 0; base < n; base += kKeysInFlight * kScanThreads) {
    K v[kKeysInFlight];
    if (base == 0) {
#pragma unroll
      for (int j = 0; j < kKeysInFlight; ++j) v[j] = held[j];
    } else {
      key_batch(keys, n, base, v);
    }
#pragma unroll
    for (int j = 0; j < kKeysInFlight; ++j) {
      const int i = base + j * kScanThreads + tid;
      const long k = static_cast<long>(v[j]) - lo;
      if (i < n) inverse[i] = (k >= 0 && k < range) ? s_table[k] : -1;
    }
  }
  return rank;
}

template <typename K>
__global__ __launch_bounds__(kScanThreads) void unique_small_kernel(const K* __restrict__ keys, int n, long lo, int range,
                                                                    K* __restrict__ unique, int64_t* __restrict__ inverse,
                                                                    int* __restrict__ n_unique) {
  extern __shared__ int s_table[];
  K held[kKeysInFlight];
  key_batch(keys, n, 0, held);
  const int count = unique_in_lds(keys, n, lo, range, held, unique, inverse, s_table);
  if (threadIdx.x == kScanThreads - 1) *n_unique = count;
}

// The same when the range is not known: the keys are read once for their smallest and largest, which go
// into found[1] and found[2]; found[0] is the number of unique keys, or -1 (nothing else written)
// where the range is more than the table holds.  Bound by latency, as is all around it: finding the range with
// library calls took three launches and a wait of the host before this one (gathering 2048 cells of 4 flows by
// their tags 243 -> 166 us).
template <typename K>
__device__ __forceinline__ void range_of_workgroup(K& lo, K& hi) {
  __shared__ K s_lo[kScanThreads / kWave], s_hi[kScanThreads / kWave];
  for (int d = 1; d < kWave; d <<= 1) lo = min(lo, __shfl_xor(lo, d, kWave)), hi = max(hi, __shfl_xor(hi, d, kWave));
  if (lane_id() == 0) s_lo[threadIdx.x >> 6] = lo, s_hi[threadIdx.x >> 6] = hi;
  __syncthreads();
  for (int w = 0; w < kScanThreads / kWave; ++w) lo = min(lo, s_lo[w]), hi = max(hi, s_hi[w]);
}

template <typename K>
__global__ __launch_bounds__(kScanThreads) void unique_whole_kernel(const K* __restrict__ keys, int n, K* __restrict__ unique,
                                                                    int64_t* __restrict__ inverse, int64_t* __restrict__ found) {
  extern __shared__ int s_table[];
  K held[kKeysInFlight];
  key_batch(keys, n, 0, held);
  K lo = held[0], hi = held[0];
  auto take = [&](const K (&v)[kKeysInFlight]) {
#pragma unroll
    for (int j = 0; j < kKeysInFlight; ++j) lo = min(lo, v[j]), hi = max(hi, v[j]);
  };
  take(held);
  for (int base = kKeysInFlight * kScanThreads; base < n; base += kKeysInFlight * kScanThreads) {
    K v[kKeysInFlight];
    key_batch(keys, n, base, v);
    take(v);
  }
  range_of_workgroup(lo, hi);
  const uint64_t span = static_cast<uint64_t>(hi) - static_cast<uint64_t>(lo);  // range - 1, whatever the signs
  const bool last = threadIdx.x == kScanThreads - 1;
  if (last) found[1] = lo, found[2] = hi;
  if (span >= kSmallRange) {
    if (last) found[0] = -1;
    return;
  }
  const int count = unique_in_lds(keys, n, static_cast<long>(lo), static_cast<int>(span) + 1, held, unique, inverse, s_table);
  if (last) found[0] = count;
}

// Pushes row p on the list of output row index[p]: head[r] is 1 + the row pushed last (0: empty),
// next[p] is 1 + the row pushed before p.  Rows with an index outside [0, n_out) are left out.
template <typename K>
__global__ void link_rows_kernel(const K* __restrict__ index, int P, int n_out, int* __restrict__ head,
                                 int* __restrict__ next) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P) return;
  const long r = static_cast<long>(index[p]);
  next[p] = (r >= 0 && r < n_out) ? atomicExch(&head[r], p + 1) : 0;
}

// The same with the clearing of the heads in the same launch: one workgroup, for inputs so small
// that every thread issues one exchange (a second launch costs more than that; beyond it the
// exchanges of one workgroup queue up behind each other).
constexpr int kSmallLinkRows = 1024, kSmallLinkOut = 4096;

template <typename K>
__global__ __launch_bounds__(kScanThreads) void clear_and_link_kernel(const K* __restrict__ index, int P,
                                                                      int n_out, int* __restrict__ head,
                                                                      int* __restrict__ next) {
  for (int r = threadIdx.x; r < n_out; r += kScanThreads) head[r] = 0;
  __syncthreads();  // the stores above have reached memory before any exchange below
  for (int p = threadIdx.x; p < P; p += kScanThreads) {
    const long r = static_cast<long>(index[p]);
    next[p] = (r >= 0 && r < n_out) ? atomicExch(&head[r], p + 1) : 0;
  }
}

// Rows that lie in several buffers, one behind the other: row p is row p - start[f] of the buffer of flow f.
constexpr int kMaxFlows = BRT_MAX_FLOWS, kFlowRows = BRT_FLOW_ROWS_MAX;
static_assert(kMaxFlows == kWave && kFlowRows == kKeysInFlight * kScanThreads, "a lane per flow, a thread's keys in registers");
struct Flows {
  const void* rows[kMaxFlows];
  int start[kMaxFlows + 1];  // start[count] and all behind it: the number of rows
  int count;
};

// Unique tags, the lists of the rows behind every one of them (as link_rows_kernel makes them) and their number, for the tags of
// several flows, in one launch of one workgroup: up to kFlowRows tags, which stay in registers, and a range that the table
// holds, which then serves as the heads of the lists.  found and its copy in host memory are {number or -1, smallest,
// largest}; a word behind the latter tells the host that it is whole.  Bound by latency.  Concatenating tags and rows, unique,
// reading its number back, clearing the heads, linking and a fill were eight launches, and 10 of 48 us of kernels went into copies of
// rows: 2048 fp32 cells of 512 elements over 4 flows, two each, scattered and gathered 101 -> 74 us.
template <typename K>
__global__ __launch_bounds__(kScanThreads) void unique_flows_kernel(Flows flows, K* __restrict__ unique, int* __restrict__ head,
                                                                    int* __restrict__ next, int* __restrict__ number,
                                                                    int64_t* __restrict__ found, int* host) {
  extern __shared__ int s_table[];
  __shared__ const K* s_rows[kMaxFlows];
  __shared__ int s_start[kMaxFlows];
  __shared__ int s_count;
  const int tid = threadIdx.x, n = flows.start[kMaxFlows];
  if (tid < kMaxFlows) {
    s_rows[tid] = static_cast<const K*>(flows.rows[tid]);
    s_start[tid] = flows.start[tid];
  }
  __syncthreads();
  K held[kKeysInFlight];
#pragma unroll
  for (int j = 0; j < kKeysInFlight; ++j) {
    const int i = min(j * kScanThreads + tid, n - 1);
    int f = 0;  // the last flow that starts at or before i: the one that holds it
#pragma unroll
    for (int step = kMaxFlows / 2; step != 0; step >>= 1) f += s_start[f + step] <= i ? step : 0;
    held[j] = s_rows[f][i - s_start[f]];
  }
  K lo = held[0], hi = held[0];
#pragma unroll
  for (int j = 1; j < kKeysInFlight; ++j) lo = min(lo, held[j]), hi = max(hi, held[j]);
  range_of_workgroup(lo, hi);
  const uint64_t span = static_cast<uint64_t>(hi) - static_cast<uint64_t>(lo);
  int count = -1;
  if (span < kSmallRange)
    count = ranks_in_lds<K>(nullptr, n, static_cast<long>(lo), static_cast<int>(span) + 1, held, unique, s_table);
  if (tid == kScanThreads - 1) {
    s_count = count;
    const int64_t out[3] = {count, static_cast<int64_t>(lo), static_cast<int64_t>(hi)};
    *number = count;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      found[i] = out[i];
      if (host != nullptr) {
        host[2 * i] = static_cast<int>(out[i]);
        host[2 * i + 1] = static_cast<int>(out[i] >> 32);
      }
    }
    if (host != nullptr) {
      __threadfence_system();
      __hip_atomic_store(host + 6, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
  if (span >= kSmallRange) return;
  int rank[kKeysInFlight];
#pragma unroll
  for (int j = 0; j < kKeysInFlight; ++j) rank[j] = s_table[static_cast<long>(held[j]) - static_cast<long>(lo)];
  __syncthreads();
  count = s_count;
  for (int r = tid; r < count; r += kScanThreads) s_table[r] = 0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kKeysInFlight; ++j) {
    const int p = j * kScanThreads + tid;
    if (p < n) next[p] = __hip_atomic_exchange(&s_table[rank[j]], p + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  __syncthreads();
  for (int r = tid; r < count; r += kScanThreads) head[r] = s_table[r];
}

struct NoFlows {};
struct SumArgs {
  const void* src;  // (FLOWS: unused)
  void* dst;
  const int* head;
  const int* next;
  int n_out, cpr;  // cpr: copy units per row
};

// One wavefront per output row.  The contributing rows are collected from the list into lanes
// (lane i holds the i-th row met), ranked against each other and moved to ascending order with
// one cross-lane permute; a list longer than a wavefront is summed by repeated search instead
// (for every next row, walk the list for the smallest row number above the last one).
// FLOWS: the rows lie in several buffers; a lane keeps the first row and the address of a flow, and the flow of a row is found
// with one ballot.
template <int BYTES, int IN_DT, int OUT_DT, bool FLOWS>
__global__ __launch_bounds__(256) void sum_rows_by_index_kernel(SumArgs a, std::conditional_t<FLOWS, Flows, NoFlows> flows) {
  using U = typename Unit<BYTES>::type;
  constexpr int NE = BYTES / elem_bytes(IN_DT);
  constexpr int OUT_BYTES = NE * elem_bytes(OUT_DT);
  constexpr int kAhead = 4;
  const int lane = lane_id();
  const int r = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (r >= a.n_out) return;
  const U* __restrict__ src = static_cast<const U*>(a.src);
  char* __restrict__ dst = static_cast<char*>(a.dst) + static_cast<size_t>(r) * a.cpr * OUT_BYTES;
  int flow_start = 0;
  uint64_t flow_rows = 0;
  if constexpr (FLOWS) {
    flow_start = flows.start[lane];
    flow_rows = reinterpret_cast<uint64_t>(flows.rows[lane]);
  }
  auto row = [&](int p) -> const U* {  // p: the same in the whole wavefront
    if constexpr (FLOWS) {
      const int f = __popcll(__ballot(flow_start <= p)) - 1;  // the last flow that starts at or before p
      const uint64_t from = static_cast<uint64_t>(static_cast<uint32_t>(read_lane(static_cast<int>(flow_rows), f))) |
                            static_cast<uint64_t>(static_cast<uint32_t>(read_lane(static_cast<int>(flow_rows >> 32), f))) << 32;
      return reinterpret_cast<const U*>(from) + static_cast<size_t>(p - read_lane(flow_start, f)) * a.cpr;
    } else {
      return src + static_cast<size_t>(p) * a.cpr;
    }
  };

  int cur = __builtin_amdgcn_readfirstlane(a.head[r]);
  int count = 0, mine = INT_MAX;
  while (cur != 0 && count < kWave) {
    if (lane == count) mine = cur - 1;
    cur = __builtin_amdgcn_readfirstlane(a.next[cur - 1]);
    ++count;
  }
  count = __builtin_amdgcn_readfirstlane(count);
  const bool longer = cur != 0;
  int ordered = mine;
  if (!longer && count > 1) {
    int below = 0;
    for (int j = 0; j < count; ++j) below += read_lane(mine, j) < mine ? 1 : 0;
    // lanes past the list all rank `count`; whichever of them lands there carries INT_MAX
    ordered = __builtin_amdgcn_ds_permute(min(below, kWave - 1) << 2, mine);
  }

  for (int off0 = 0; off0 < a.cpr; off0 += kWave) {
    const int off = off0 + lane;
    const bool live = off < a.cpr;
    float acc[NE];
#pragma unroll
    for (int q = 0; q < NE; ++q) acc[q] = 0.0f;
    if (!longer) {
      for (int i0 = 0; i0 < count; i0 += kAhead) {
        U val[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
          if (i0 + u < count) {
            const U* const from = row(read_lane(ordered, i0 + u));
            if (live) val[u] = from[off];
          }
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
          if (i0 + u < count && live) {
            float x[NE];
            unpack<IN_DT, BYTES>(val[u], x);
#pragma unroll
            for (int q = 0; q < NE; ++q) acc[q] += x[q];
          }
        }
      }
    } else {
      int last = -1;
      while (true) {
        int best = INT_MAX;
        for (int c = __builtin_amdgcn_readfirstlane(a.head[r]); c != 0;
             c = __builtin_amdgcn_readfirstlane(a.next[c - 1])) {
          const int p = c - 1;
          if (p > last && p < best) best = p;
        }
        if (best == INT_MAX) break;
        last = best;
        const U* const from = row(best);
        if (live) {
          float x[NE];
          unpack<IN_DT, BYTES>(from[off], x);
#pragma unroll
          for (int q = 0; q < NE; ++q) acc[q] += x[q];
        }
      }
    }
    // streamed when not widening and the rows are whole 16-byte units (the case of the expert
    // outputs this op exists for); narrower units mean short or odd rows, better merged in the L2
    if (live) pack_store<OUT_DT, NE, IN_DT == OUT_DT && BYTES == 16>(dst + static_cast<size_t>(off) * OUT_BYTES, acc);
  }
}

template <int IN_DT, int OUT_DT, typename F = NoFlows>
void launch_sum(int unit, const SumArgs& a, hipStream_t st, const F& flows = {}) {
  const dim3 grid((a.n_out + 3) / 4), block(256);
  constexpr bool kFlows = std::is_same_v<F, Flows>;
  if (unit == 16) hipLaunchKernelGGL((sum_rows_by_index_kernel<16, IN_DT, OUT_DT, kFlows>), grid, block, 0, st, a, flows);
  else if (unit == 8) hipLaunchKernelGGL((sum_rows_by_index_kernel<8, IN_DT, OUT_DT, kFlows>), grid, block, 0, st, a, flows);
  else if (unit == 4) hipLaunchKernelGGL((sum_rows_by_index_kernel<4, IN_DT, OUT_DT, kFlows>), grid, block, 0, st, a, flows);
  else if constexpr (IN_DT != BRT_F32)
    hipLaunchKernelGGL((sum_rows_by_index_kernel<2, IN_DT, OUT_DT, kFlows>), grid, block, 0, st, a, flows);
}

// The flows of a launch: false where a row count is negative, a flow with rows has no address, or they are too many.
bool collect_flows(const void* const* rows, const int32_t* counts, int flow_num, Flows* out) {
  if (rows == nullptr || counts == nullptr || flow_num < 1 || flow_num > kMaxFlows) return false;
  long start = 0;
  for (int f = 0; f < flow_num; ++f) {
    if (counts[f] < 0 || (counts[f] > 0 && rows[f] == nullptr)) return false;
    out->rows[f] = rows[f];
    out->start[f] = static_cast<int>(start);
    start += counts[f];
    if (start > INT_MAX) return false;
  }
  for (int f = flow_num; f < kMaxFlows; ++f) out->rows[f] = nullptr;
  for (int f = flow_num; f <= kMaxFlows; ++f) out->start[f] = static_cast<int>(start);
  out->count = flow_num;
  return true;
}

long scan_blocks(long range) { return (range + kScanChunk - 1) / kScanChunk; }

}  // namespace
}  // namespace brt

using namespace brt;

extern "C" size_t brt_hip_unique_tags_workspace_bytes(long lo, long hi) {
  if (hi < lo) return 16;
  const long range = hi - lo + 1;
  if (range > kMaxRange) return 0;
  return static_cast<size_t>(range + scan_blocks(range)) * sizeof(int) + 16;
}

extern "C" int brt_hip_unique_tags(const void* tags, int tag_bits, long n, long lo, long hi,
                                   void* workspace, size_t workspace_bytes, void* unique_tags,
                                   int64_t* inverse, int32_t* n_unique, void* stream) {
  if (tag_bits != 32 && tag_bits != 64) return fail(BRT_E_INVALID, "tag_bits must be 32 or 64, got %d", tag_bits);
  if (n < 0 || hi < lo) return fail(BRT_E_INVALID, "bad arguments n=%ld lo=%ld hi=%ld", n, lo, hi);
  if (!n_unique) return fail(BRT_E_INVALID, "null n_unique");
  hipStream_t st = as_stream(stream);
  const long range = hi - lo + 1;
  if (range > kMaxRange)
    return fail(BRT_E_UNSUPPORTED, "tag range %ld exceeds %ld", range, kMaxRange);
  if (!tags || !workspace || !unique_tags || !inverse) return fail(BRT_E_INVALID, "null argument");
  const size_t need = brt_hip_unique_tags_workspace_bytes(lo, hi);
  if (workspace_bytes < need || !aligned(workspace, 4))
    return fail(BRT_E_INVALID, "workspace of %zu bytes, need %zu", workspace_bytes, need);
  if (range <= kSmallRange && n >= 1 && n <= kSmallCount) {  // (no keys: the general path below)
    const size_t lds = static_cast<size_t>(range) * sizeof(int);
    const void* fn = tag_bits == 32 ? reinterpret_cast<const void*>(&unique_small_kernel<int32_t>)
                                    : reinterpret_cast<const void*>(&unique_small_kernel<int64_t>);
    if (const int rc = allow_dynamic_lds(fn, kSmallRange * static_cast<int>(sizeof(int))); rc != BRT_OK) return rc;
    if (tag_bits == 32)
      hipLaunchKernelGGL(unique_small_kernel<int32_t>, dim3(1), dim3(kScanThreads), lds, st,
                         static_cast<const int32_t*>(tags), static_cast<int>(n), lo, static_cast<int>(range),
                         static_cast<int32_t*>(unique_tags), inverse, n_unique);
    else
      hipLaunchKernelGGL(unique_small_kernel<int64_t>, dim3(1), dim3(kScanThreads), lds, st,
                         static_cast<const int64_t*>(tags), static_cast<int>(n), lo, static_cast<int>(range),
                         static_cast<int64_t*>(unique_tags), inverse, n_unique);
    return check_launch("unique_small_kernel");
  }
  int* table = static_cast<int*>(workspace);
  const long blocks = scan_blocks(range);
  int* totals = table + range;
  hipLaunchKernelGGL(fill_zero_kernel, dim3(static_cast<unsigned>((range + 255) / 256)), dim3(256), 0, st,
                     table, range);
  if (n > 0) {
    const dim3 grid(static_cast<unsigned>((n + 255) / 256)), block(256);
    if (tag_bits == 32)
      hipLaunchKernelGGL(mark_present_kernel<int32_t>, grid, block, 0, st,
                         static_cast<const int32_t*>(tags), n, lo, range, table);
    else
      hipLaunchKernelGGL(mark_present_kernel<int64_t>, grid, block, 0, st,
                         static_cast<const int64_t*>(tags), n, lo, range, table);
  }
  if (blocks > 1)
    hipLaunchKernelGGL(chunk_total_kernel, dim3(static_cast<unsigned>(blocks)), dim3(kScanThreads), 0, st,
                       table, range, totals);
  if (tag_bits == 32)
    hipLaunchKernelGGL(rank_emit_kernel<int32_t>, dim3(static_cast<unsigned>(blocks)), dim3(kScanThreads), 0,
                       st, table, range, totals, lo, static_cast<int32_t*>(unique_tags), n_unique);
  else
    hipLaunchKernelGGL(rank_emit_kernel<int64_t>, dim3(static_cast<unsigned>(blocks)), dim3(kScanThreads), 0,
                       st, table, range, totals, lo, static_cast<int64_t*>(unique_tags), n_unique);
  if (n > 0) {
    const dim3 grid(static_cast<unsigned>((n + 255) / 256)), block(256);
    if (tag_bits == 32)
      hipLaunchKernelGGL(inverse_kernel<int32_t>, grid, block, 0, st, static_cast<const int32_t*>(tags), n,
                         lo, range, table, inverse);
    else
      hipLaunchKernelGGL(inverse_kernel<int64_t>, grid, block, 0, st, static_cast<const int64_t*>(tags), n,
                         lo, range, table, inverse);
  }
  return check_launch("unique_tags");
}

extern "C" int brt_hip_unique_tags_whole(const void* tags, int tag_bits, long n, void* unique_tags, int64_t* inverse,
                                         int64_t* found, void* stream) {
  if (tag_bits != 32 && tag_bits != 64) return fail(BRT_E_INVALID, "tag_bits must be 32 or 64, got %d", tag_bits);
  if (n < 1) return fail(BRT_E_INVALID, "bad arguments n=%ld", n);
  if (n > kSmallCount) return fail(BRT_E_UNSUPPORTED, "more than %ld tags", kSmallCount);
  if (!tags || !unique_tags || !inverse || !found) return fail(BRT_E_INVALID, "null argument");
  const int lds = kSmallRange * static_cast<int>(sizeof(int));
  const bool narrow = tag_bits == 32;
  const void* fn = narrow ? reinterpret_cast<const void*>(&unique_whole_kernel<int32_t>)
                          : reinterpret_cast<const void*>(&unique_whole_kernel<int64_t>);
  if (const int rc = allow_dynamic_lds(fn, lds); rc != BRT_OK) return rc;
  if (narrow)
    hipLaunchKernelGGL(unique_whole_kernel<int32_t>, dim3(1), dim3(kScanThreads), lds, as_stream(stream),
                       static_cast<const int32_t*>(tags), static_cast<int>(n), static_cast<int32_t*>(unique_tags), inverse, found);
  else
    hipLaunchKernelGGL(unique_whole_kernel<int64_t>, dim3(1), dim3(kScanThreads), lds, as_stream(stream),
                       static_cast<const int64_t*>(tags), static_cast<int>(n), static_cast<int64_t*>(unique_tags), inverse, found);
  return check_launch("unique_whole_kernel");
}

extern "C" int brt_hip_unique_tags_of_flows(const void* const* tags, const int32_t* rows, int flow_num, int tag_bits, void* unique_tags,
                                            int32_t* head, int32_t* next, int32_t* n_unique, int64_t* found, int32_t* host,
                                            void* stream) {
  if (tag_bits != 32 && tag_bits != 64) return fail(BRT_E_INVALID, "tag_bits must be 32 or 64, got %d", tag_bits);
  Flows flows;
  if (!collect_flows(tags, rows, flow_num, &flows)) return fail(BRT_E_INVALID, "bad flows (%d of them)", flow_num);
  const int n = flows.start[kMaxFlows];
  if (n < 1) return fail(BRT_E_INVALID, "no tags");
  if (n > kFlowRows) return fail(BRT_E_UNSUPPORTED, "more than %d tags", kFlowRows);
  if (!unique_tags || !head || !next || !n_unique || !found) return fail(BRT_E_INVALID, "null argument");
  for (int f = 0; f < flow_num; ++f)
    if (!aligned(tags[f], tag_bits / 8)) return fail(BRT_E_INVALID, "tags are not aligned to their size");
  const int lds = kSmallRange * static_cast<int>(sizeof(int));
  const bool narrow = tag_bits == 32;
  const void* fn = narrow ? reinterpret_cast<const void*>(&unique_flows_kernel<int32_t>)
                          : reinterpret_cast<const void*>(&unique_flows_kernel<int64_t>);
  if (const int rc = allow_dynamic_lds(fn, lds); rc != BRT_OK) return rc;
  if (narrow)
    hipLaunchKernelGGL(unique_flows_kernel<int32_t>, dim3(1), dim3(kScanThreads), lds, as_stream(stream), flows,
                       static_cast<int32_t*>(unique_tags), head, next, n_unique, found, host);
  else
    hipLaunchKernelGGL(unique_flows_kernel<int64_t>, dim3(1), dim3(kScanThreads), lds, as_stream(stream), flows,
                       static_cast<int64_t*>(unique_tags), head, next, n_unique, found, host);
  return check_launch("unique_flows_kernel");
}

extern "C" int brt_hip_combine_flows(const void* const* in_data, const int32_t* rows, int flow_num, void* out_data, const int32_t* head,
                                     const int32_t* next, int cell, int n_out, int dtype, void* stream) {
  if (cell < 0 || n_out < 0) return fail(BRT_E_INVALID, "bad shape cell=%d n_out=%d", cell, n_out);
  if (dtype != BRT_F32 && dtype != BRT_F16 && dtype != BRT_BF16) return fail(BRT_E_UNSUPPORTED, "dtype %d", dtype);
  Flows flows;
  if (!collect_flows(in_data, rows, flow_num, &flows)) return fail(BRT_E_INVALID, "bad flows (%d of them)", flow_num);
  if (n_out == 0 || cell == 0) return BRT_OK;
  if (!out_data || !head || !next) return fail(BRT_E_INVALID, "null argument");
  const int es = elem_bytes(dtype);
  const size_t row_bytes = static_cast<size_t>(cell) * es;
  uintptr_t address = reinterpret_cast<uintptr_t>(out_data);
  for (int f = 0; f < flow_num; ++f)
    if (rows[f] > 0) address |= reinterpret_cast<uintptr_t>(in_data[f]);
  int unit = 0;
  for (int b = 16; b >= es && unit == 0; b >>= 1)
    if (row_bytes % b == 0 && address % b == 0) unit = b;
  if (unit == 0) return fail(BRT_E_INVALID, "rows are not aligned to their element size");
  const SumArgs a{nullptr, out_data, head, next, n_out, static_cast<int>(row_bytes / unit)};
  if (dtype == BRT_F32) launch_sum<BRT_F32, BRT_F32>(unit, a, as_stream(stream), flows);
  else if (dtype == BRT_F16) launch_sum<BRT_F16, BRT_F16>(unit, a, as_stream(stream), flows);
  else launch_sum<BRT_BF16, BRT_BF16>(unit, a, as_stream(stream), flows);
  return check_launch("combine_flows");
}

extern "C" size_t brt_hip_combine_by_index_workspace_bytes(int P, int n_out) {
  return (static_cast<size_t>(std::max(P, 0)) + static_cast<size_t>(std::max(n_out, 0))) * sizeof(int) + 16;
}

extern "C" int brt_hip_combine_by_index(const void* in_data, void* out_data, const void* index,
                                        int index_bits, int P, int cell, int n_out, void* workspace,
                                        size_t workspace_bytes, int in_dtype, int out_dtype,
                                        void* stream) {
  if (index_bits != 32 && index_bits != 64)
    return fail(BRT_E_INVALID, "index_bits must be 32 or 64, got %d", index_bits);
  if (P < 0 || cell < 0 || n_out < 0) return fail(BRT_E_INVALID, "bad shape P=%d cell=%d n_out=%d", P, cell, n_out);
  const bool same = in_dtype == out_dtype;
  const bool widen = (in_dtype == BRT_F16 || in_dtype == BRT_BF16) && out_dtype == BRT_F32;
  if ((in_dtype != BRT_F32 && in_dtype != BRT_F16 && in_dtype != BRT_BF16) || !(same || widen))
    return fail(BRT_E_UNSUPPORTED, "dtype pair %d -> %d", in_dtype, out_dtype);
  if (n_out == 0 || cell == 0) return BRT_OK;
  if (!out_data || !workspace || (P > 0 && (!in_data || !index))) return fail(BRT_E_INVALID, "null argument");
  const size_t need = brt_hip_combine_by_index_workspace_bytes(P, n_out);
  if (workspace_bytes < need || !aligned(workspace, 4))
    return fail(BRT_E_INVALID, "workspace of %zu bytes, need %zu", workspace_bytes, need);
  const int es = elem_bytes(in_dtype), os = elem_bytes(out_dtype);
  const size_t row_bytes = static_cast<size_t>(cell) * es;
  int unit = 0;
  for (int b = 16; b >= es && unit == 0; b >>= 1)
    if (row_bytes % b == 0 && aligned(in_data, b) && aligned(out_data, std::min(16, b * os / es))) unit = b;
  if (unit == 0) return fail(BRT_E_INVALID, "rows are not aligned to their element size");
  hipStream_t st = as_stream(stream);
  int* head = static_cast<int*>(workspace);
  int* next = head + n_out;
  const bool small = P <= kSmallLinkRows && n_out <= kSmallLinkOut;
  if (small) {
    if (index_bits == 32)
      hipLaunchKernelGGL(clear_and_link_kernel<int32_t>, dim3(1), dim3(kScanThreads), 0, st,
                         static_cast<const int32_t*>(index), P, n_out, head, next);
    else
      hipLaunchKernelGGL(clear_and_link_kernel<int64_t>, dim3(1), dim3(kScanThreads), 0, st,
                         static_cast<const int64_t*>(index), P, n_out, head, next);
  } else {
    hipLaunchKernelGGL(fill_zero_kernel, dim3((n_out + 255) / 256), dim3(256), 0, st, head, static_cast<long>(n_out));
  }
  if (P > 0 && !small) {
    const dim3 grid((P + 255) / 256), block(256);
    if (index_bits == 32)
      hipLaunchKernelGGL(link_rows_kernel<int32_t>, grid, block, 0, st, static_cast<const int32_t*>(index), P,
                         n_out, head, next);
    else
      hipLaunchKernelGGL(link_rows_kernel<int64_t>, grid, block, 0, st, static_cast<const int64_t*>(index), P,
                         n_out, head, next);
  }
  SumArgs a{in_data, out_data, head, next, n_out, static_cast<int>(row_bytes / unit)};
  if (in_dtype == BRT_F32) launch_sum<BRT_F32, BRT_F32>(unit, a, st);
  else if (in_dtype == BRT_F16 && same) launch_sum<BRT_F16, BRT_F16>(unit, a, st);
  else if (in_dtype == BRT_F16) launch_sum<BRT_F16, BRT_F32>(unit, a, st);
  else if (same) launch_sum<BRT_BF16, BRT_BF16>(unit, a, st);
  else launch_sum<BRT_BF16, BRT_F32>(unit, a, st);
  return check_launch("combine_by_index");
}
