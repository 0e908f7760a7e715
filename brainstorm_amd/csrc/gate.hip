// Gate front-end: scores -> int32 hot mask with ones at the k largest scores of every row.
//
// Replaces the three torch launches of the reference's TopKProtocol
// (python/brt/router/protocol/topk.py:26-31: torch.topk, zeros_like, scatter_) with one pass
// that reads the scores once and writes the mask once.  Order of torch.topk: NaN above every
// number; among equal scores (which torch leaves unspecified) the lowest column wins.
//
// Lanes are columns.  Up to 32 columns: a wavefront takes 64/ep rows per step (ep = columns
// rounded up to a power of two) and every selection is a butterfly max inside the row's lane
// segment plus a ballot that picks the lowest lane holding the maximum.  More than 32 columns:
// every lane keeps the columns lane, lane+64, ... of up to four rows in registers.
//
// The compact form of the same pass writes, instead of (or beside) the dense mask, the k chosen
// columns of every row in the order of selection and their weights: the scores themselves, or
// their softmax over the row (fp32: exp(x - max) / sum, the front end of the Switch router,
// benchmark/switch_moe/switch_transformer.py:240-253, and of the Swin-MoE gate,
// python/brt/router/protocol/swin_moe.py:100-107).  k words per row instead of E.
#include <algorithm>

#include "common.hpp"
#include "gate.hpp"

namespace brt {
namespace {

constexpr int kBlock = 256;
constexpr int kMaxPerLane = 16;  // columns per lane in the wide path: up to 1024 columns

struct GateArgs {
  const void* scores;
  int* mask;       // [T, E] or null
  int* ids;        // [T, k] chosen columns in the order of selection (compact form only)
  float* weights;  // [T, k] or null
  int softmax;     // weights are the softmax of the row instead of the scores
  int T, E, k;
  int ep_shift;  // log2 of the lane segment of a row (E <= 64)
  int rows_pw;   // rows per wavefront
};

template <int DT, bool COMPACT>
__global__ __launch_bounds__(kBlock) void topk_mask_kernel(GateArgs a) {
  const int lane = threadIdx.x & (kWave - 1);
  const long wave = static_cast<long>(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int ep = 1 << a.ep_shift, rps = kWave >> a.ep_shift;
  const int e = lane & (ep - 1), sub = lane >> a.ep_shift;
  const unsigned long long seg = (ep == kWave ? ~0ull : ((1ull << ep) - 1ull)) << (sub * ep);
  const long t0 = wave * a.rows_pw;
  const int nt = static_cast<int>(max(0l, min(static_cast<long>(a.rows_pw), a.T - t0)));
  for (int r0 = 0; r0 < nt; r0 += rps) {
    const int row = r0 + sub;
    const bool live = row < nt && e < a.E;
    const float x = live ? load_score<DT>(a.scores, static_cast<size_t>(t0 + row) * a.E + e) : 0.0f;
    uint32_t key = live ? score_key(x) : 0u;
    float weight = x;
    if (COMPACT && a.softmax) {
      const float top = segment_max(live ? x : -INFINITY, ep);
      const float ex = live ? expf(x - top) : 0.0f;
      weight = ex / segment_sum(ex, ep);
    }
    int taken = 0;
    for (int pass = 0; pass < a.k; ++pass) {
      const uint32_t best = segment_max(key, ep);
      const unsigned long long tied = __ballot(key == best && key != 0) & seg;
      if (tied != 0 && lane == __builtin_ctzll(tied)) {
        taken = 1;
        key = 0;
        if (COMPACT) {
          const size_t slot = static_cast<size_t>(t0 + row) * a.k + pass;
          a.ids[slot] = e;
          if (a.weights) a.weights[slot] = weight;
        }
      }
    }
    if (live && (!COMPACT || a.mask)) a.mask[static_cast<size_t>(t0 + row) * a.E + e] = taken;
  }
}

// More than 32 columns: PER of them a lane (column c * 64 + lane), ROWS rows at a time, whose loads travel together and
// whose selections are independent of each other.  A selection is the wavefront's maximum, taken on the DPP network, and
// one ballot per 64 columns, searched for the lowest bit on the scalar unit.  Bound by memory with one path a row, by
// the issue of the selections with more.  fp32 scores -> mask: 131072 x 128, one path 57.1 us with 16 columns a lane,
// one row at a time and butterflies -> 19.9 (6.7 TB/s), 131072 x 100, four paths 126 -> 29, 20000 x 256 12.5 -> 7.7,
// 16384 x 1000 32.4 -> 20.8; 131072 x 64, for which the kernel above was used, 17.4 -> 12.9, four paths 36.3 -> 21.4.
// Up to 32 columns several rows share a wavefront above, and 131072 x 32 takes 12.5.
template <int DT, bool COMPACT, int PER, int ROWS>
__global__ __launch_bounds__(kBlock) void topk_mask_wide_kernel(GateArgs a) {
  const int lane = threadIdx.x & (kWave - 1);
  const long wave = static_cast<long>(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const long t0 = wave * a.rows_pw;
  const int nt = static_cast<int>(max(0l, min(static_cast<long>(a.rows_pw), a.T - t0)));
  for (int r0 = 0; r0 < nt; r0 += ROWS) {
    uint32_t key[ROWS][PER];
    float weight[ROWS][PER];
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
      for (int c = 0; c < PER; ++c)  // (clamped, not guarded: a guarded load waits for the one before)
        weight[r][c] = load_score<DT>(a.scores, static_cast<size_t>(t0 + min(r0 + r, nt - 1)) * a.E +
                                                    min(c * kWave + lane, a.E - 1));
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
      for (int c = 0; c < PER; ++c) {
        const bool live = c * kWave + lane < a.E;
        if (!live) weight[r][c] = -INFINITY;
        key[r][c] = live ? score_key(weight[r][c]) : 0u;
      }
    if (COMPACT && a.softmax) {
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        float top = -INFINITY;
#pragma unroll
        for (int c = 0; c < PER; ++c) top = fmaxf(top, weight[r][c]);
        top = segment_max(top, kWave);
        float sum = 0.0f;
#pragma unroll
        for (int c = 0; c < PER; ++c) {
          weight[r][c] = weight[r][c] == -INFINITY ? 0.0f : expf(weight[r][c] - top);
          sum += weight[r][c];
        }
        sum = segment_sum(sum, kWave);
#pragma unroll
        for (int c = 0; c < PER; ++c) weight[r][c] = weight[r][c] / sum;
      }
    }
    for (int pass = 0; pass < a.k; ++pass) {
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        uint32_t mine = 0;
#pragma unroll
        for (int c = 0; c < PER; ++c) mine = max(mine, key[r][c]);
        const uint32_t best = wave_max(mine);
        // lowest column holding the maximum: lowest c first, then lowest lane
        unsigned long long searched = 0;  // columns found so far: only the first one is taken
#pragma unroll
        for (int c = 0; c < PER; ++c) {
          const unsigned long long tied = searched ? 0ull : __ballot(key[r][c] == best && best != 0);
          searched |= tied;
          if (__ffsll(tied) - 1 == lane) {
            key[r][c] = 0;  // taken
            if (COMPACT && r0 + r < nt) {
              const size_t slot = static_cast<size_t>(t0 + r0 + r) * a.k + pass;
              a.ids[slot] = c * kWave + lane;
              if (a.weights) a.weights[slot] = weight[r][c];
            }
          }
        }
      }
    }
    if (!COMPACT || a.mask) {
#pragma unroll
      for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int c = 0; c < PER; ++c) {
          const int col = c * kWave + lane;
          if (r0 + r < nt && col < a.E) a.mask[static_cast<size_t>(t0 + r0 + r) * a.E + col] = key[r][c] == 0;
        }
    }
  }
}

}  // namespace
}  // namespace brt

using namespace brt;

namespace {

int launch_gate(GateArgs a, int dtype, bool compact, void* stream) {
  const int T = a.T, E = a.E, k = a.k;
  if (T < 0 || E <= 0 || k < 0 || k > E) return fail(BRT_E_INVALID, "bad shape T=%d E=%d k=%d", T, E, k);
  if (dtype != BRT_F32 && dtype != BRT_F16 && dtype != BRT_BF16)
    return fail(BRT_E_UNSUPPORTED, "dtype %d is not supported", dtype);
  if (E > kWave * kMaxPerLane) return fail(BRT_E_UNSUPPORTED, "more than %d paths", kWave * kMaxPerLane);
  if (static_cast<long>(T) * E >= (1l << 31)) return fail(BRT_E_UNSUPPORTED, "T*E >= 2^31");
  if (T == 0) return BRT_OK;
  if (!a.scores || (compact ? (k > 0 && !a.ids) : !a.mask)) return fail(BRT_E_INVALID, "null argument");
  int shift = 0;
  while ((1 << shift) < std::min(E, kWave)) ++shift;
  a.ep_shift = shift;
  const int rps = E <= kWave ? kWave >> shift : 1;
  // about 8192 wavefronts (the chip a few times over), whole steps per wavefront: a wavefront's
  // steps run one after the other, each a full memory round trip
  long rows = ((T + 8191) / 8192 + rps - 1) / rps * rps;
  if (E > kWave / 2 && E <= 4 * kWave && rows > 1) rows = (rows + 3) / 4 * 4;  // whole steps of the wide kernel
  rows = std::min<long>(std::max<long>(rows, rps), 16l * rps);
  a.rows_pw = static_cast<int>(rows);
  const long n_waves = (T + a.rows_pw - 1) / a.rows_pw;
  const int waves_pb = kBlock / kWave;
  const dim3 grid(static_cast<unsigned>((n_waves + waves_pb - 1) / waves_pb)), block(kBlock);
  hipStream_t st = as_stream(stream);
// 8192 rows and fewer are one a wavefront; a step of several rows would only repeat the last
#define BRT_GATE_WIDE(DT, COMPACT, PER, ROWS)                                                                   \
  if (a.rows_pw == 1) hipLaunchKernelGGL((topk_mask_wide_kernel<DT, COMPACT, PER, 1>), grid, block, 0, st, a); \
  else hipLaunchKernelGGL((topk_mask_wide_kernel<DT, COMPACT, PER, ROWS>), grid, block, 0, st, a);
#define BRT_GATE_KERNELS(DT, COMPACT)                                                               \
  if (E <= kWave / 2) hipLaunchKernelGGL((topk_mask_kernel<DT, COMPACT>), grid, block, 0, st, a);   \
  else if (E <= kWave) { BRT_GATE_WIDE(DT, COMPACT, 1, 4) }                                         \
  else if (E <= 2 * kWave) { BRT_GATE_WIDE(DT, COMPACT, 2, 4) }                                     \
  else if (E <= 4 * kWave) { BRT_GATE_WIDE(DT, COMPACT, 4, 2) }                                     \
  else hipLaunchKernelGGL((topk_mask_wide_kernel<DT, COMPACT, kMaxPerLane, 1>), grid, block, 0, st, a);
#define BRT_GATE_LAUNCH(DT)                   \
  if (compact) { BRT_GATE_KERNELS(DT, true) } \
  else { BRT_GATE_KERNELS(DT, false) }
  if (dtype == BRT_F32) { BRT_GATE_LAUNCH(BRT_F32) }
  else if (dtype == BRT_F16) { BRT_GATE_LAUNCH(BRT_F16) }
  else { BRT_GATE_LAUNCH(BRT_BF16) }
#undef BRT_GATE_WIDE
#undef BRT_GATE_LAUNCH
#undef BRT_GATE_KERNELS
  return check_launch("topk_mask_kernel");
}

}  // namespace

extern "C" int brt_hip_topk_hot_mask(const void* scores, int32_t* hot_mask, int T, int E, int k,
                                     int dtype, void* stream) {
  GateArgs a{};
  a.scores = scores; a.mask = hot_mask; a.T = T; a.E = E; a.k = k;
  return launch_gate(a, dtype, false, stream);
}

extern "C" int brt_hip_gate_topk(const void* scores, int T, int E, int k, int dtype, int softmax,
                                 int32_t* path_ids, float* weights, int32_t* hot_mask, void* stream) {
  GateArgs a{};
  a.scores = scores; a.mask = hot_mask; a.ids = path_ids; a.weights = weights;
  a.softmax = softmax; a.T = T; a.E = E; a.k = k;
  return launch_gate(a, dtype, true, stream);
}
