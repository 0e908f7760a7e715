// Grouped expert GEMM, third kernel: few rows per expert and few tiles (decode batches, small layers),
// where the weights have to be streamed by as many CUs as there are and nothing else costs anything.
//
// Same contract as grouped_gemm.hip (out[rows of e] = act(x[rows of e] @ W_e^T + b_e), one launch,
// loads read on the device; reference: src/jit/compiler.cu:151-246).  What differs:
//
//   - A workgroup owns XR rows x 32 * NT columns, a tile so small that even a contracting GEMM of a
//     few experts has a workgroup per CU, and its S wavefronts split K between them: each multiplies its
//     own slice of K for the whole tile, and the partial sums meet in LDS at the end, added in
//     wavefront order (the result does not depend on timing).
//     Every tile shape splits K the same way, so a row's bits do not depend on the shape.
//   - A wavefront's K loop is its own: operands go from global memory straight into its corner of
//     LDS (a ring of D K-steps of 64, whole 128-byte lines per row, swizzled on the global side as
//     in grouped_gemm_pingpong.hip), waits count its own loads, and there is no barrier.
//     A deep ring matters less than many wavefronts with requests in flight: two or three workgroups
//     share a CU.
//   - Rows past the expert's load and past N address past the buffer extent: zeros, no request.
//   - Every wavefront finds the tile by itself (DPP scan + ballot over the loads, the weight
//     pointers fetched in the same round trip), so the first weight request leaves two round trips
//     after the start.  Gathered rows add one, which the weight requests do not wait for.
#include <algorithm>

#include "common.hpp"
#include "grouped_gemm.hpp"
#include "rows.hpp"

namespace brt {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

constexpr int kBK = 64;
constexpr int kRowB = kBK * 2;                 // bytes of one operand row in one stage: one cache line
constexpr int kSub = kBK / 16;                 // MFMA k-steps per stage
constexpr uint32_t kOutOfRange = 0x80000000u;  // buffer offset past any extent: reads as zero

__device__ __forceinline__ i32x4 make_rsrc(const void* p, size_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  i32x4 r;
  r[0] = static_cast<int>(a);
  r[1] = static_cast<int>((a >> 32) & 0xffff);
  r[2] = static_cast<int>(bytes > 0x7fffffffull ? 0x7fffffffull : bytes);
  r[3] = 0x00020000;
  return r;
}

// 16 / 4 bytes per lane from the buffer straight into LDS at lds_base + 16 (4) * lane; every wait for
// such a load is written out below
__device__ __forceinline__ void load_to_lds(const i32x4& rsrc, uint32_t voffset, uint32_t soffset, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"(__builtin_amdgcn_readfirstlane(lds_base)), "v"(voffset), "s"(rsrc), "s"(__builtin_amdgcn_readfirstlane(soffset))
               : "memory");
}
__device__ __forceinline__ void load_word_to_lds(const i32x4& rsrc, uint32_t voffset, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dword %1, %2, 0 offen lds"
               :
               : "s"(lds_base), "v"(voffset), "s"(rsrc)
               : "memory");
}

template <int N>
__device__ __forceinline__ void wait_loads_but() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }
// waits until at most `left` of this wavefront's loads are outstanding (rounded down to an even number)
__device__ __forceinline__ void wait_loads(int left) {
  switch (left >> 1) {
#define BRT_WAIT(n) case n: wait_loads_but<2 * n>(); break;
    BRT_WAIT(1) BRT_WAIT(2) BRT_WAIT(3) BRT_WAIT(4) BRT_WAIT(5) BRT_WAIT(6) BRT_WAIT(7) BRT_WAIT(8)
    BRT_WAIT(9) BRT_WAIT(10) BRT_WAIT(11) BRT_WAIT(12) BRT_WAIT(13) BRT_WAIT(14) BRT_WAIT(15) BRT_WAIT(16)
    BRT_WAIT(17) BRT_WAIT(18) BRT_WAIT(19) BRT_WAIT(20) BRT_WAIT(21) BRT_WAIT(22) BRT_WAIT(23) BRT_WAIT(24)
#undef BRT_WAIT
    default: wait_loads_but<0>();
  }
}
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory"); }

template <int XR, int NT, int S, int D>
struct Shape {
  static constexpr int kXi = XR / 8, kWi = NT * 4;             // load instructions of one K-step: rows of x, weight rows
  static constexpr int kStage = (kXi + kWi) * 1024;
  static constexpr int kBN = NT * 32;
  static constexpr int kSumRow = kBN * 4 + 16;                 // padded row of a partial sum
  static constexpr int kRing = D * kStage > XR * kSumRow ? D * kStage : XR * kSumRow;
  static constexpr int kLds = S * kRing;
  static_assert(XR % 32 == 0, "whole MFMA row tiles");
  static_assert(D * (kXi + kWi) <= 48, "the waits count up to 48 loads");
};

template <int XR, int NT, int S, int D, int ACT, bool ROUTED, bool OUTF32>
__global__ __launch_bounds__(S * 64) void grouped_gemm_skinny_kernel(GemmArgs a) {
  using H = Shape<XR, NT, S, D>;
  constexpr int MT = XR / 32;
  constexpr int kXi = H::kXi, kWi = H::kWi, kL = kXi + kWi;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int K = a.K;

  // ---- which tile: column tiles of a row block are consecutive, so they spread over the XCDs -----
  const int block = blockIdx.x / a.tiles_n, n0 = (blockIdx.x - block * a.tiles_n) * H::kBN;
  int e = -1, row0 = 0, rows = 0, seat0 = 0, carry_t = 0, carry_m = 0;
  const __bf16* w_e = nullptr;
  for (int base = 0; base < a.E; base += kWave) {
    const int el = base + lane;
    const int m = el < a.E ? a.loads[el] : 0;
    const uint64_t wp = el < a.E ? reinterpret_cast<uint64_t>(a.w[el]) : 0;
    const int blocks = (m + XR - 1) / XR;
    const int incl_t = wave_inclusive_scan(blocks), incl_m = wave_inclusive_scan(m);
    const int first = carry_t + incl_t - blocks;
    const unsigned long long hit = __ballot(block >= first && block < first + blocks);
    if (hit != 0) {
      const int src = __builtin_ctzll(hit);
      const int local = block - read_lane(first, src);
      e = base + src;
      seat0 = local * XR;
      row0 = carry_m + read_lane(incl_m - m, src) + seat0;
      rows = min(min(XR, read_lane(m, src) - seat0), a.P - row0);
      w_e = reinterpret_cast<const __bf16*>(static_cast<uint64_t>(static_cast<uint32_t>(read_lane(static_cast<int>(wp), src))) |
                                            static_cast<uint64_t>(static_cast<uint32_t>(read_lane(static_cast<int>(wp >> 32), src))) << 32);
      break;
    }
    carry_t += read_lane(incl_t, kWave - 1);
    carry_m += read_lane(incl_m, kWave - 1);
  }
  if (e < 0) {
    // Row blocks past the last one clear the tags of the rows no path owns, XR rows each: the grid
    // holds P / XR + min(E, P) of them (rounded up), the experts use at most (total + (XR - 1) * used experts) / XR.
    if (ROUTED && a.row_tags_out != nullptr && n0 == 0) {
      const long r = static_cast<long>(carry_m) + static_cast<long>(block - carry_t) * XR + tid;
      if (tid < XR && r < a.P) a.row_tags_out[r] = 0;
    }
    return;
  }

  // ---- this wavefront's slice of K: at least two K-steps ------------------------------------------
  const int k_tiles = (K + kBK - 1) / kBK;
  const int per = max(2, (k_tiles + S - 1) / S);
  const int parts = (k_tiles + per - 1) / per;  // wavefronts that have one
  const int kt0 = wave * per, n = __builtin_amdgcn_readfirstlane(min(per, k_tiles - kt0));
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem))) + wave * H::kRing;
  char* const ring = smem + wave * H::kRing;

  f32x16 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x16{};

  if (n > 0) {
    // Lane l lands at slot l & 7 of row l >> 3 of the 8 rows a load fills and fetches chunk
    // slot ^ ((row >> 1) & 7) of that row; a chunk past K (the last K-step only) reads as zero.
    const bool gather = ROUTED && a.gather != 0;
    const i32x4 res_w = make_rsrc(w_e + static_cast<size_t>(n0) * K, static_cast<size_t>(a.N - n0) * K * 2);
    const i32x4 res_x = gather ? make_rsrc(a.x, static_cast<size_t>(a.T) * K * 2)
                               : make_rsrc(a.x + static_cast<size_t>(row0) * K, static_cast<size_t>(a.P - row0) * K * 2);
    const int r8 = lane >> 3;
    const int chunk0 = (lane & 7) ^ (r8 >> 1);  // even groups of 8 rows; odd ones flip bit 2
    uint32_t off_w[kWi], off_x[kXi];
#pragma unroll
    for (int i = 0; i < kWi; ++i) {
      const int row = i * 8 + r8;
      off_w[i] = n0 + row < a.N ? (static_cast<uint32_t>(row) * K + (chunk0 ^ ((i & 1) << 2)) * 8) * 2 : kOutOfRange;
    }
    const int tail_chunks = K % kBK != 0 ? (K % kBK) / 8 : 8;  // chunks of the last K-step that exist
    auto fetch = [&](const i32x4& res, uint32_t off, int i, int kt, uint32_t to) {
      if (kt == k_tiles - 1 && (chunk0 ^ ((i & 1) << 2)) >= tail_chunks) off = kOutOfRange;
      load_to_lds(res, off, kt * kRowB, to);
    };
    auto load_w = [&](int s) {
      const uint32_t to = lds0 + (s % D) * H::kStage;
#pragma unroll
      for (int i = 0; i < kWi; ++i) fetch(res_w, off_w[i], i, kt0 + s, to + i * 1024);
    };
    auto load_x = [&](int s) {
      const uint32_t to = lds0 + (s % D) * H::kStage + kWi * 1024;
#pragma unroll
      for (int i = 0; i < kXi; ++i) fetch(res_x, off_x[i], i, kt0 + s, to + i * 1024);
    };
    const int primed = min(D, n);
    if (gather) {
      // The words that name the rows land in the last stage's room for x (a direct load, so that
      // waiting for it does not wait for the weight requests behind it).
      const int last = D - 1;
      const uint32_t words = lds0 + last * H::kStage + kWi * 1024;
      const bool slot_ok = lane < rows && (a.tag_vector || seat0 + lane < a.T);
      const size_t first = a.tag_vector ? static_cast<size_t>(row0) : static_cast<size_t>(seat0) * a.E + e;
      const i32x4 res_t = make_rsrc(a.tags + first, static_cast<size_t>(XR) * (a.tag_vector ? 1 : a.E) * 4);
      load_word_to_lds(res_t, slot_ok ? static_cast<uint32_t>(lane) * (a.tag_vector ? 1 : a.E) * 4 : kOutOfRange, words);
      for (int s = 0; s < primed; ++s) load_w(s);
      wait_loads(primed * kWi);
#pragma unroll
      for (int i = 0; i < kXi; ++i) {
        const int word = *reinterpret_cast<const volatile int*>(ring + last * H::kStage + kWi * 1024 + (i * 8 + r8) * 4);
        const int cell = cell_of_word(a, word);
        off_x[i] = cell >= 0 ? (static_cast<uint32_t>(cell) * K + (chunk0 ^ ((i & 1) << 2)) * 8) * 2 : kOutOfRange;
      }
      wait_lds();
      for (int s = 0; s < primed; ++s) load_x(s);
    } else {
#pragma unroll
      for (int i = 0; i < kXi; ++i) {
        const int row = i * 8 + r8;
        off_x[i] = row < rows ? (static_cast<uint32_t>(row) * K + (chunk0 ^ ((i & 1) << 2)) * 8) * 2 : kOutOfRange;
      }
      for (int s = 0; s < primed; ++s) load_w(s), load_x(s);
    }

    // MFMA operand: this lane feeds row (lane % 32), k-half (lane / 32) of a 32 x 16 block
    const int frag_row = lane & 31, frag_k = lane >> 5;
    const int swz = (frag_row >> 1) & 7;
    const int frag_w = frag_row * kRowB;
    const int frag_x = kWi * 1024 + frag_row * kRowB;
    for (int s = 0; s < n; ++s) {
      // loads issued after the last one of K-step s
      int younger = min(D - 1, n - 1 - s) * kL;
      if (gather && s < primed) younger = (primed - 1 - s) * kXi + min(s, max(n - D, 0)) * kL;
      wait_loads(younger);
      const char* const at = ring + (s % D) * H::kStage;
      bf16x8 fw[kSub][NT], fx[kSub][MT];
#pragma unroll
      for (int ks = 0; ks < kSub; ++ks) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
          fw[ks][j] = *reinterpret_cast<const bf16x8*>(at + frag_w + j * 32 * kRowB + (((ks * 2 + frag_k) ^ swz) << 4));
#pragma unroll
        for (int i = 0; i < MT; ++i)
          fx[ks][i] = *reinterpret_cast<const bf16x8*>(at + frag_x + i * 32 * kRowB + (((ks * 2 + frag_k) ^ swz) << 4));
      }
      wait_lds();  // the fragments are in registers: the slot may be filled again
      if (s + D < n) load_w(s + D), load_x(s + D);
#pragma unroll
      for (int ks = 0; ks < kSub; ++ks)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw[ks][j], fx[ks][i], acc[i][j], 0, 0, 0);
    }

    // partial sums into this wavefront's ring (every load has landed): element r of tile (i, j) is
    // row 32 i + lane % 32, column 32 j + 8 * (r / 4) + 4 * (lane / 32) + r % 4
#pragma unroll
    for (int i = 0; i < MT; ++i) {
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<f32x4*>(ring + (i * 32 + frag_row) * H::kSumRow + (j * 32 + 8 * g + 4 * frag_k) * 4) =
              f32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
    }
  }
  __syncthreads();

  // ---- sum over the wavefronts, bias, activation ---------------------------------------------------
  auto column_sum = [&](int r, int c) {  // one output element (accumulate form)
    float v = 0.0f;
    for (int s = 0; s < parts; ++s) {
      const float p = reinterpret_cast<const float*>(smem + s * H::kRing + r * H::kSumRow)[c];
      v = s == 0 ? p : v + p;
    }
    return apply_act<ACT>(v + (a.bias != nullptr ? static_cast<float>(a.bias[e][n0 + c]) : 0.0f));
  };
  if constexpr (ROUTED && !OUTF32) {
    if (a.gates != nullptr) {  // acc_out[cell] += gate * bf16(row), as in grouped_gemm.hip
      for (int q = tid; q < rows * H::kBN; q += S * 64) {
        const int r = q / H::kBN, c = q - r * H::kBN;
        const int cell = routed_cell(a, e, row0 + r, seat0 + r);
        if (cell < 0 || n0 + c >= a.N) continue;
        const size_t at = a.tag_vector ? static_cast<size_t>(a.tags[row0 + r]) - 1 : static_cast<size_t>(cell) * a.E + e;
        const float v = static_cast<float>(static_cast<__bf16>(column_sum(r, c)));
        unsafeAtomicAdd(a.acc_out + static_cast<size_t>(cell) * a.N + n0 + c, v * a.gates[at]);
      }
      return;
    }
  }
  // 8 columns of one row per thread and step: 16-byte stores (two of them for fp32)
  constexpr int kChunks = H::kBN / 8;
  for (int q = tid; q < rows * kChunks; q += S * 64) {
    const int r = q / kChunks, c = q - r * kChunks;
    if (n0 + c * 8 >= a.N) continue;
    long to = row0 + r;
    if (ROUTED && (a.scatter || a.row_tags_out != nullptr)) {
      const int cell = routed_cell(a, e, row0 + r, seat0 + r);
      // side output for a combine that runs later: written once per row block
      if (a.row_tags_out != nullptr && n0 == 0 && c == 0) a.row_tags_out[row0 + r] = cell + 1;
      if (a.scatter) to = cell;
    }
    if (to < 0) continue;
    float v[8];
    for (int s = 0; s < parts; ++s) {
      const float* const from = reinterpret_cast<const float*>(smem + s * H::kRing + r * H::kSumRow) + c * 8;
#pragma unroll
      for (int w = 0; w < 8; ++w) v[w] = s == 0 ? from[w] : v[w] + from[w];
    }
    const __bf16* const bias = a.bias != nullptr ? a.bias[e] + n0 + c * 8 : nullptr;
#pragma unroll
    for (int w = 0; w < 8; ++w) v[w] = apply_act<ACT>(v[w] + (bias != nullptr ? static_cast<float>(bias[w]) : 0.0f));
    if constexpr (OUTF32) {
      f32x4* const o = reinterpret_cast<f32x4*>(a.out_f32 + static_cast<size_t>(to) * a.N + n0 + c * 8);
      // -0 -> +0, as a combine would
      o[0] = f32x4{v[0] + 0.0f, v[1] + 0.0f, v[2] + 0.0f, v[3] + 0.0f};
      o[1] = f32x4{v[4] + 0.0f, v[5] + 0.0f, v[6] + 0.0f, v[7] + 0.0f};
    } else {
      u32x4 o;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        o[w] = float_to_bf16(v[2 * w]) | (float_to_bf16(v[2 * w + 1]) << 16);
        if (ROUTED && a.scatter) o[w] = plus_zero<BRT_BF16>(o[w]);  // the combine adds the row to zero
      }
      *reinterpret_cast<u32x4*>(a.out + static_cast<size_t>(to) * a.N + n0 + c * 8) = o;
    }
  }
}

template <int XR, int NT, int S, int D, int ACT, bool ROUTED, bool OUTF32>
int launch(GemmArgs& a, hipStream_t st) {
  using H = Shape<XR, NT, S, D>;
  a.tiles_n = (a.N + H::kBN - 1) / H::kBN;
  // the sum over experts of ceil(M_e / XR) never exceeds P / XR + min(E, P)
  const long blocks = (static_cast<long>(a.P) + XR - 1) / XR + std::min(a.E, a.P);
  auto* fn = &grouped_gemm_skinny_kernel<XR, NT, S, D, ACT, ROUTED, OUTF32>;
  if (const int rc = allow_dynamic_lds(reinterpret_cast<const void*>(fn), H::kLds); rc != BRT_OK) return rc;
  hipLaunchKernelGGL(fn, dim3(static_cast<unsigned>(blocks * a.tiles_n)), dim3(S * 64), H::kLds, st, a);
  return check_launch("grouped_gemm_skinny_kernel");
}

template <int XR, int NT, int S, int D, int ACT>
int launch_form(GemmArgs& a, hipStream_t st) {
  const bool f32 = a.out_f32 != nullptr;
  if (a.tags != nullptr) return f32 ? launch<XR, NT, S, D, ACT, true, true>(a, st) : launch<XR, NT, S, D, ACT, true, false>(a, st);
  return f32 ? launch<XR, NT, S, D, ACT, false, true>(a, st) : launch<XR, NT, S, D, ACT, false, false>(a, st);
}

template <int XR, int NT, int S, int D>
int launch_act(GemmArgs& a, int act, hipStream_t st) {
  if (act == BRT_ACT_GELU) return launch_form<XR, NT, S, D, BRT_ACT_GELU>(a, st);
  if (act == BRT_ACT_RELU) return launch_form<XR, NT, S, D, BRT_ACT_RELU>(a, st);
  return launch_form<XR, NT, S, D, BRT_ACT_NONE>(a, st);
}

}  // namespace

// Where this kernel is taken, against the 160-row kernel.  Both were timed on 2 to 200 rows per expert,
// 4 to 128 experts, 512 <-> 2048, 768 <-> 3072, 1024 <-> 4096, 2048 <-> 8192 and 320 <-> 640; the
// rule gives up small gains rather than lose where the 160-row kernel is the faster one.
//   - Up to 28 rows per expert (one row block): while the weights are less than 0.3 GB (8 experts x 3 rows
//     3072 -> 768: 43.9 -> 9.7 us, 32 x 8 rows 4096 -> 1024 68.3 -> 46.3 us).  Beyond, the wide tiles stream
//     them at the memory's rate (32 x 19 rows 6656 -> 1664, 709 MB: 113 us there, 129 us here; 32 x 16 rows
//     1920 -> 3840, 472 MB: 75.5 and 84.0 us), except where they cannot: half of the CUs without a
//     tile (16 x 12 rows 6656 -> 1664 89.6 -> 66.7 us), a K whose rows lie multiples of 4 KB apart (64 x 16
//     rows 4096 -> 1024 119 -> 91 us) or experts of which many get no row at all (128 experts, 183 rows
//     896 -> 3584 124 -> 96 us); up to 1 GB (32 x 8 rows 8192 -> 2048, 1.07 GB: 171 us there, 200 us here).
//   - More rows: every block of 32 or 64 rows streams the weights again (from the L2), which pays
//     while the 160-row kernel has too few 160 x 256 tiles for the CUs: up to 72 of them, however many
//     rows that are (8 x 120 rows 3072 -> 768 46.9 -> 22.4 us, 4 x 1300 rows 1024 -> 256 24.5 -> 12.3 us,
//     32 x 120 rows 2048 -> 512 36.6 -> 36.2 us; not 64 x 120 rows, 128 tiles: 44.9 -> 59.9 us), and up to
//     160 for few experts of up to 128 rows and 0.15 GB (4 x 120 rows 2048 -> 8192 77.2 -> 43.0 us; not 16 x 40
//     rows 3840 -> 1920, 236 MB: 55.9 -> 72.5 us).
bool skinny_gemm_applies(const GemmArgs& a) {
  const long used = std::min(a.E, a.P);
  const long tiles = std::max<long>((a.P + 159) / 160, used) * ((a.N + 255) / 256);
  const double weight_bytes = 2.0 * used * a.N * a.K;
  if (tiles <= 72) return true;
  if (a.P <= 28 * used) {
    if (weight_bytes < 3e8) return true;
    return weight_bytes < 1e9 && (tiles <= 128 || a.K % 2048 == 0 || 2l * a.P <= 3 * used);
  }
  return a.P <= 128 * used && tiles <= 160 && a.E <= 16 && weight_bytes < 1.5e8;
}

// Shape of the tile.  Few workgroups: the narrowest one, so that every CU gets one (at most 264 of 32 x
// 64).  Else 64 columns, which read the activation rows half as often; 64 rows where experts have
// more than 64 (the weights are streamed half as often).  A long K with few rows (K = 3072, 24 rows,
// 8 experts: 11.1 us against 15.4 us) stays on the narrow tile, whose two stages keep loads in flight.
int launch_skinny_gemm(GemmArgs& a, int act, hipStream_t st) {
  const long used = std::min(a.E, a.P);
  const double rows = static_cast<double>(a.P) / used;
  const bool narrow = used * std::max(1.0, rows / 32 + 0.5) * a.N / 64 <= 264 || (rows <= 40 && a.K > 1536);
  if (narrow) return launch_act<32, 1, 4, 2>(a, act, st);
  if (rows <= 40 || (rows <= 64 && a.K <= 1024)) return launch_act<32, 2, 4, 1>(a, act, st);
  return launch_act<64, 2, 4, 1>(a, act, st);
}

}  // namespace brt
