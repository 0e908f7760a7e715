// Grouped expert GEMM, third kernel: few rows per expert and few tiles (decode batches, small layers),
// where the weights have to be streamed by as many CUs as there are and nothing else costs anything.
//
// Same contract as grouped_gemm.hip (out[rows of e] = act(x[rows of e] @ W_e^T + b_e), one launch,
// loads read on the device; reference: src/jit/compiler.cu:151-246), and the same bits: the products of an
// output element are summed in order of K by the same instruction in all three kernels, so that a
// row does not depend on which of them the number of rows selects.  What differs:
//
//   - A workgroup owns XR rows x 32 * NT columns, a tile so small that even a contracting GEMM of a
//     few experts has a workgroup per CU.  One wavefront per 32 x 32 block multiplies it over all of K;
//     all four load.
//   - Operands go from global memory straight into LDS (a ring of D K-steps of 64, whole 128-byte lines
//     per row, swizzled on the global side as in grouped_gemm_pingpong.hip).  Every wavefront loads a quarter
//     of each K-step, waits for its own part of the next one and meets the others at one
//     barrier per K-step, behind which that K-step can be read and the stage of the one being
//     multiplied be filled again.
//   - Bound by the chain of K-steps where tiles are few: four dependent MFMAs and the fragment reads of the
//     next K-step, which run behind them; about 170 ns per K-step (8 experts x 3 rows 3072 -> 768:
//     11.2 us; the four wavefronts summing a quarter of K each, which gives other bits, 10.7 us; one
//     wavefront that loads by itself 18.7 us).  K-steps of 128 with half the barriers change nothing.
//   - Rows past the expert's load and past N address past the buffer extent: zeros, no request.
//   - fp32 rows of x (X32) are loaded as they are and rounded to bf16 on their way from LDS to the matrix unit: the cast
//     kernel and its pass over the rows go (figures at the choice of the tile).
//   - Every wavefront finds the tile by itself (DPP scan + ballot over the loads, the weight
//     pointers fetched in the same round trip), so the first weight request leaves two round trips
//     after the start.  Gathered rows add one, which the weight requests do not wait for.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "grouped_gemm.hpp"
#include "rows.hpp"

namespace brt {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
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
// waits until at most `left` of this wavefront's loads are outstanding; left <= MOST (the fewer cases, the shorter the branches:
// cases up to 16 for every tile cost the shortest chains 0.2 us, 4 x 8 rows 520 -> 1032 5.5 us for 5.3)
template <int MOST>
__device__ __forceinline__ void wait_loads(int left) {
  switch (left) {
#define BRT_WAIT(n) case n: if constexpr (n <= MOST) { wait_loads_but<n>(); break; } else { __builtin_unreachable(); }
    BRT_WAIT(1) BRT_WAIT(2) BRT_WAIT(3) BRT_WAIT(4) BRT_WAIT(5) BRT_WAIT(6) BRT_WAIT(7) BRT_WAIT(8)
    BRT_WAIT(9) BRT_WAIT(10) BRT_WAIT(11) BRT_WAIT(12) BRT_WAIT(13) BRT_WAIT(14) BRT_WAIT(15) BRT_WAIT(16)
#undef BRT_WAIT
    default: wait_loads_but<0>();
  }
}
// lgkmcnt(0) alone, known to the compiler (which counts on behind it)
__device__ __forceinline__ void wait_lds() {
  __builtin_amdgcn_s_waitcnt(0xc07f);
  asm volatile("" : : : "memory");
}

constexpr int kWaves = 4;
constexpr int kXcds = 8;

template <int XR, int NT, int D, bool X32>
struct Shape {
  static constexpr int kXRowB = X32 ? 2 * kRowB : kRowB;       // bytes of one row of x in one stage
  static constexpr int kXRows = 1024 / kXRowB;                 // rows of x that one load instruction fills
  static constexpr int kXi = XR / kXRows, kWi = NT * 4;        // load instructions of one K-step: rows of x, weight rows
  static constexpr int kXw = kXi / kWaves, kWw = kWi / kWaves;  // ... of one wavefront
  static constexpr int kStage = (kXi + kWi) * 1024;
  static constexpr int kBN = NT * 32;
  static constexpr int kSumRow = kBN * 4 + 16;                 // padded row of the sums on their way out
  static constexpr int kLds = D * kStage > XR * kSumRow ? D * kStage : XR * kSumRow;
  static constexpr int kMost = (D - 1) * (kXw + kWw) > D * kWw ? (D - 1) * (kXw + kWw) : D * kWw;  // most loads a wait leaves out
  static_assert(XR % 32 == 0 && XR / 32 * NT <= kWaves, "at most one 32 x 32 block per wavefront");
  static_assert(D >= 2 && kMost <= 16, "the waits count up to 16 loads");
};

template <int XR, int NT, int D, int ACT, bool ROUTED, bool OUTF32, bool X32>
__global__ __launch_bounds__(kWaves * kWave) void grouped_gemm_skinny_kernel(GemmArgs a) {
  using H = Shape<XR, NT, D, X32>;
  constexpr int kXB = X32 ? 4 : 2;  // bytes of one element of x
  constexpr int kWi = H::kWi, kXw = H::kXw, kWw = H::kWw, kL = kXw + kWw;
  constexpr int kBlocks = XR / 32 * NT;  // 32 x 32 blocks of the tile, one wavefront each
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int K = a.K;

  // ---- which tile: an entry of the list of tiles (experts, their row blocks, column tiles).  The workgroups go to the XCDs in
  // turn, so in the order of the list the column tiles of a row block spread over the XCDs; in patch order every XCD takes an
  // eighth of the list, whose rows of x it reads alone.
  int m = lane < a.E ? a.loads[lane] : 0;
  uint64_t wp = lane < a.E ? reinterpret_cast<uint64_t>(a.w[lane]) : 0;
  auto row_blocks = [](int rows_of_e) { return (rows_of_e + XR - 1) / XR; };
  int block, column, idle = 0;  // idle: behind which many workgroups without a tile this one stands
  if (a.patch) {
    int total = read_lane(wave_inclusive_scan(row_blocks(m)), kWave - 1);
    for (int base = kWave; base < a.E; base += kWave)
      total += read_lane(wave_inclusive_scan(base + lane < a.E ? row_blocks(a.loads[base + lane]) : 0), kWave - 1);
    const int tiles = min(total, a.tiles_m_max) * a.tiles_n, share = (tiles + kXcds - 1) / kXcds;
    const int xcd = blockIdx.x % kXcds, turn = blockIdx.x / kXcds;
    const int before = min(xcd * share, tiles), own = min(share, tiles - before);
    const unsigned tile = before + turn;
    block = __umulhi(tile, a.tiles_n_inverse), column = tile - block * a.tiles_n;
    if (column >= a.tiles_n) ++block, column -= a.tiles_n;
    if (turn >= own) block = total, column = 0, idle = xcd * (gridDim.x / kXcds) - before + turn - own;
  } else {
    block = blockIdx.x / a.tiles_n, column = blockIdx.x - block * a.tiles_n;
  }
  const int n0 = column * H::kBN;
  int e = -1, row0 = 0, rows = 0, seat0 = 0, carry_t = 0, carry_m = 0;
  const __bf16* w_e = nullptr;
  for (int base = 0; base < a.E; base += kWave) {
    if (base != 0) {
      m = base + lane < a.E ? a.loads[base + lane] : 0;
      wp = base + lane < a.E ? reinterpret_cast<uint64_t>(a.w[base + lane]) : 0;
    }
    const int blocks = row_blocks(m);
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
      const long r = static_cast<long>(carry_m) + static_cast<long>(block - carry_t + idle) * XR + tid;
      if (tid < XR && r < a.P) a.row_tags_out[r] = 0;
    }
    return;
  }

  const int k_tiles = (K + kBK - 1) / kBK;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem)));

  // ---- this wavefront's loads: row groups of 8 rows, kWw of the weights and kXw of x ----------------
  // Lane l lands at slot l & 7 of row l >> 3 of the 8 rows a load fills and fetches chunk
  // slot ^ ((row >> 1) & 7) of that row; a chunk past K (the last K-step only) reads as zero.
  const bool gather = ROUTED && a.gather != 0;
  const i32x4 res_w = make_rsrc(w_e + static_cast<size_t>(n0) * K, static_cast<size_t>(a.N - n0) * K * 2);
  const char* const x_b = reinterpret_cast<const char*>(a.x);
  const i32x4 res_x = gather ? make_rsrc(x_b, static_cast<size_t>(a.T) * K * kXB)
                             : make_rsrc(x_b + static_cast<size_t>(row0) * K * kXB, static_cast<size_t>(a.P - row0) * K * kXB);
  const int r8 = lane >> 3;
  const int first_w = wave * kWw, first_x = wave * kXw;  // row groups
  auto chunk = [&](int group) { return (lane & 7) ^ (r8 >> 1) ^ ((group & 1) << 2); };
  // fp32 rows of x are 16 chunks of 4 elements: lane l lands at slot l & 15 of row l >> 4 and fetches chunk slot ^ (row & 15)
  const int rx = X32 ? lane >> 4 : r8;
  auto chunk_x = [&](int group) { return X32 ? (lane & 15) ^ ((group * 4 + rx) & 15) : chunk(group); };
  uint32_t off_w[kWw], off_x[kXw];
#pragma unroll
  for (int i = 0; i < kWw; ++i) {
    const int row = (first_w + i) * 8 + r8;
    off_w[i] = n0 + row < a.N ? (static_cast<uint32_t>(row) * K + chunk(first_w + i) * 8) * 2 : kOutOfRange;
  }
  const int tail_chunks = K % kBK != 0 ? (K % kBK) / 8 : 8;  // chunks of the last K-step that exist
  auto fetch = [&](const i32x4& res, uint32_t off, bool past, int s, int step, uint32_t to) {
    if (s == k_tiles - 1 && past) off = kOutOfRange;
    load_to_lds(res, off, s * step, to);
  };
  auto load_w = [&](int s, uint32_t stage, int i) {
    fetch(res_w, off_w[i], chunk(first_w + i) >= tail_chunks, s, kRowB, lds0 + stage + (first_w + i) * 1024);
  };
  auto load_x = [&](int s, uint32_t stage, int i) {
    fetch(res_x, off_x[i], chunk_x(first_x + i) >= (X32 ? 2 : 1) * tail_chunks, s, H::kXRowB, lds0 + stage + (kWi + first_x + i) * 1024);
  };
  const int primed = min(D, k_tiles);
  if (gather) {
    // The words that name this wavefront's rows land in the last stage's room for them (a direct load, so
    // that waiting for it does not wait for the weight requests behind it).
    const uint32_t words = (D - 1) * H::kStage + (kWi + first_x) * 1024;
    const int row = first_x * H::kXRows + lane;
    const bool slot_ok = lane < kXw * H::kXRows && row < rows && (a.tag_vector || seat0 + row < a.T);
    const size_t first = a.tag_vector ? static_cast<size_t>(row0) : static_cast<size_t>(seat0) * a.E + e;
    const i32x4 res_t = make_rsrc(a.tags + first, static_cast<size_t>(XR) * (a.tag_vector ? 1 : a.E) * 4);
    load_word_to_lds(res_t, slot_ok ? static_cast<uint32_t>(row) * (a.tag_vector ? 1 : a.E) * 4 : kOutOfRange, lds0 + words);
    for (int s = 0; s < primed; ++s)
#pragma unroll
      for (int i = 0; i < kWw; ++i) load_w(s, s * H::kStage, i);
    wait_loads<H::kMost>(primed * kWw);
#pragma unroll
    for (int i = 0; i < kXw; ++i) {
      const int word = *reinterpret_cast<const volatile int*>(smem + words + (i * H::kXRows + rx) * 4);
      const int cell = cell_of_word(a, word);
      off_x[i] = cell >= 0 ? static_cast<uint32_t>(cell) * K * kXB + chunk_x(first_x + i) * 16 : kOutOfRange;
    }
    wait_lds();
    for (int s = 0; s < primed; ++s)
#pragma unroll
      for (int i = 0; i < kXw; ++i) load_x(s, s * H::kStage, i);
  } else {
#pragma unroll
    for (int i = 0; i < kXw; ++i) {
      const int row = (first_x + i) * H::kXRows + rx;
      off_x[i] = row < rows ? static_cast<uint32_t>(row) * K * kXB + chunk_x(first_x + i) * 16 : kOutOfRange;
    }
    for (int s = 0; s < primed; ++s) {
#pragma unroll
      for (int i = 0; i < kWw; ++i) load_w(s, s * H::kStage, i);
#pragma unroll
      for (int i = 0; i < kXw; ++i) load_x(s, s * H::kStage, i);
    }
  }

  // ---- K loop ----------------------------------------------------------------------------------------
  // MFMA operand: this lane feeds row (lane % 32), k-half (lane / 32) of a 32 x 16 block
  const bool multiplies = wave < kBlocks;
  const int block_x = wave / NT, block_w = wave % NT;
  const int frag_row = lane & 31, frag_k = lane >> 5;
  const int swz = (frag_row >> 1) & 7;
  const char* const from_w = smem + (block_w * 32 + frag_row) * kRowB;
  const char* const from_x = smem + kWi * 1024 + (block_x * 32 + frag_row) * H::kXRowB;
  struct Frags {
    bf16x8 w[kSub];
    std::conditional_t<X32, f32x8, bf16x8> x[kSub];
  };
  // fp32 rows are rounded to bf16 on their way from LDS (to nearest even, as the cast kernel does)
  auto x_of = [](const Frags& f, int ks) {
    if constexpr (X32) return __builtin_convertvector(f.x[ks], bf16x8);
    else return f.x[ks];
  };
  auto read_frags = [&](Frags& f, uint32_t stage, int ks) {
    const uint32_t at = stage + (((ks * 2 + frag_k) ^ swz) << 4);
    f.w[ks] = *reinterpret_cast<const bf16x8*>(from_w + at);
    if constexpr (X32) {
      const int c = (ks * 2 + frag_k) * 2, swz_x = frag_row & 15;
      const f32x4 lo = *reinterpret_cast<const f32x4*>(from_x + stage + ((c ^ swz_x) << 4));
      const f32x4 hi = *reinterpret_cast<const f32x4*>(from_x + stage + (((c + 1) ^ swz_x) << 4));
      f.x[ks] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    } else {
      f.x[ks] = *reinterpret_cast<const bf16x8*>(from_x + at);
    }
  };
  // this wavefront's loads issued after the last one of K-step s, once K-steps up to `issued` have been requested
  auto younger = [&](int s, int issued) {
    return gather && s < primed ? (primed - 1 - s) * kXw + max(issued + 1 - primed, 0) * kL : (issued - s) * kL;
  };
  f32x16 acc = {};
  // K-step s, whose stage every wavefront has read: the loads of s + D go there.  A multiplying wavefront has
  // its fragments in `cur`; those of s + 1 come out of the next stage meanwhile (no branch around the reads:
  // the compiler would wait for all of them in front of every MFMA; behind the last K-step they
  // read words that nothing uses).
  using Yes = std::integral_constant<bool, true>;
  using No = std::integral_constant<bool, false>;
  uint32_t stage = 0;
  auto step = [&](const Frags& cur, Frags& next, int s, auto multiply, auto fills) {
    constexpr bool kMultiply = decltype(multiply)::value, kFills = decltype(fills)::value;
    const uint32_t ahead = stage + H::kStage == D * H::kStage ? 0 : stage + H::kStage;
    if (kFills && !(gather && s < primed)) wait_loads_but<(D - 2) * kL>();
    else if (s + 1 < k_tiles) wait_loads<H::kMost>(younger(s + 1, min(s + D, k_tiles) - 1));
    __builtin_amdgcn_s_barrier();
    if (!kFills && s + D < k_tiles) {
#pragma unroll
      for (int i = 0; i < kL; ++i) i < kWw ? load_w(s + D, stage, i) : load_x(s + D, stage, i - kWw);
    }
#pragma unroll
    for (int ks = 0; ks < kSub; ++ks) {
      if constexpr (kMultiply) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur.w[ks], x_of(cur, ks), acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        read_frags(next, ahead, ks);
      }
      if constexpr (kFills) {
#pragma unroll
        for (int i = ks * kL / kSub; i < (ks + 1) * kL / kSub; ++i) i < kWw ? load_w(s + D, stage, i) : load_x(s + D, stage, i - kWw);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (kMultiply) wait_lds();  // behind the next barrier the stage of s + 1 may be filled again
    stage = ahead;
  };
  auto k_loop = [&](auto multiply) {
    Frags f0, f1;
    wait_loads<H::kMost>(younger(0, primed - 1));
    __builtin_amdgcn_s_barrier();
    if constexpr (decltype(multiply)::value) {
#pragma unroll
      for (int ks = 0; ks < kSub; ++ks) read_frags(f0, 0, ks);
      wait_lds();
    }
    int s = 0;
    for (; s + 1 + D < k_tiles; s += 2) {
      step(f0, f1, s, multiply, Yes{});
      step(f1, f0, s + 1, multiply, Yes{});
    }
    for (; s < k_tiles; s += 2) {
      step(f0, f1, s, multiply, No{});
      if (s + 1 < k_tiles) step(f1, f0, s + 1, multiply, No{});
    }
  };
  if (multiplies) k_loop(Yes{});
  else k_loop(No{});

  // The sums into LDS (behind the last barrier nothing reads or fills the stages): element r of a block is
  // its row lane % 32, column 8 * (r / 4) + 4 * (lane / 32) + r % 4
  if (multiplies) {
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(smem + (block_x * 32 + frag_row) * H::kSumRow + (block_w * 32 + 8 * g + 4 * frag_k) * 4) =
          f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
  }
  __syncthreads();

  // ---- bias, activation ---------------------------------------------------
  auto column_sum = [&](int r, int c) {  // one output element (accumulate form)
    const float v = reinterpret_cast<const float*>(smem + r * H::kSumRow)[c];
    return apply_act<ACT>(v + (a.bias != nullptr ? static_cast<float>(a.bias[e][n0 + c]) : 0.0f));
  };
  if constexpr (ROUTED && !OUTF32) {
    if (a.gates != nullptr) {  // acc_out[cell] += gate * bf16(row), as in grouped_gemm.hip
      for (int q = tid; q < rows * H::kBN; q += kWaves * kWave) {
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
  for (int q = tid; q < rows * kChunks; q += kWaves * kWave) {
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
    const float* const from = reinterpret_cast<const float*>(smem + r * H::kSumRow) + c * 8;
#pragma unroll
    for (int w = 0; w < 8; ++w) v[w] = from[w];
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

// Estimated tiles of `block` x 64 of the result; an expert's last row block is taken as half full.
double narrow_tiles(const GemmArgs& a, int block) {
  const long used = std::min(a.E, a.P);
  const double rows = static_cast<double>(a.P) / used;
  return used * (rows > block ? rows / block + 0.5 : 1.0) * ((a.N + 63) / 64);
}

// Where the tiles are dealt in patch order.  In the order of the list every XCD's L2 draws all rows of x: eight times their bytes, beside
// weights that come once.  Dealt by expert they come once too: 12 x 95 rows 1280 -> 320 10.9 -> 7.4 us, 8 x 97 rows 4160 -> 1040
// 36.5 -> 27.6, 16 x 64 fp32 rows 2048 -> 512 17.0 -> 13.9.  Taken where the seven copies saved are a good part of the bytes (8 times the rows of x
// a fifth of the weights or more), of contracting shapes of more than one row block per expert and a tile for most CUs.  Of 74
// drawn shapes that it takes the mean is 1.18 times as fast in patch order, 3 are more than 2 % slower: weight rows 8 KB apart (8 x 115 skewed
// rows 4096 -> 1024 32.9 and 36.2).  Not taken: few tiles, which pay 0.1 us more for finding theirs (4 x 104 rows 768 -> 768 5.9 and 6.1),
// large expanding shapes, whose output lines and weights the XCDs then write and read far apart (4 x 120 rows 2048 -> 8192 42 and 46), and
// weights of 0.14 GB, of part-filled lines 40 MB, or more, likewise (16 x 123 rows 3008 -> 1504 54 and 57, 16 x 60 rows 2096 -> 1048 31 and 34).
bool experts_stay_on_an_xcd(const GemmArgs& a) {
  const long used = std::min(a.E, a.P);
  return a.N <= a.K && a.P > 32 * used && 2.0 * used * a.N * a.K < (a.K % kBK == 0 ? 1.4e8 : 4e7) && narrow_tiles(a, 32) >= 150 &&
         (a.x_f32 ? 16.0 : 8.0) * a.P >= 0.2 * used * a.N;
}

// Tiles of the 160-row kernel, 256 columns wide.
long wide_tiles(const GemmArgs& a) {
  return std::max<long>((a.P + 159) / 160, std::min(a.E, a.P)) * ((a.N + 255) / 256);
}

// Expanding shapes of 65 to 400 rows per expert that are taken because they are dealt in patch order too: with few and small tiles the 160-row
// kernel is as slow as its busiest CU, and up to 40 MB of weights stay near (us, 160-row kernel and this one: 32 x 163 rows
// 256 -> 1024 31 and 14, 64 x 94 rows 128 -> 256 15 and 5.6, 12 x 233 rows 576 -> 2304 41 and 23, 24 x 322 rows 192 -> 768 12.4 and 12.2).  Of 80 other
// drawn shapes the mean is 1.52 times as fast, three are slower (24 x 174 skewed rows 576 -> 1152 19.3 and 21.1).
// Only where the rows are whole lines; not with fewer experts (8 x 343 rows 960 -> 1920 26.1 and 26.5), more weights (24 x 124 rows 512 -> 2048, 50 MB, 18.7 and 23.1) or
// more tiles (128 x 120 rows 128 -> 512, 256 of them, 13.3 and 17.4).  Up to 96 tiles of up to 32 experts are this kernel's in any case (below)
// and stay in the order of the list.  (Dealt as well, 60 drawn ones take 0.95 of the
// time in the mean, from 0.60 -- 21 x 225 rows 384 -> 576 13.3 and 7.9 -- to 1.02.)
bool expanding_and_dealt(const GemmArgs& a) {
  const long used = std::min(a.E, a.P), tiles = wide_tiles(a);
  return a.N > a.K && a.K % kBK == 0 && used >= 12 && a.P > 64 * used && a.P <= 400 * used && tiles <= 170 && (tiles > 96 || used > 32) &&
         2.0 * used * a.N * a.K <= 4e7;
}

template <int XR, int NT, int D, int ACT, bool ROUTED, bool OUTF32, bool X32>
int launch(GemmArgs& a, hipStream_t st) {
  using H = Shape<XR, NT, D, X32>;
  a.tiles_n = (a.N + H::kBN - 1) / H::kBN;
  a.tiles_n_inverse = 0xffffffffu / static_cast<uint32_t>(a.tiles_n);
  // the sum over experts of ceil(M_e / XR) never exceeds P / XR + min(E, P)
  const long blocks = (static_cast<long>(a.P) + XR - 1) / XR + std::min(a.E, a.P);
  a.tiles_m_max = static_cast<int>(blocks);
  a.patch = experts_stay_on_an_xcd(a) || expanding_and_dealt(a);
  auto* fn = &grouped_gemm_skinny_kernel<XR, NT, D, ACT, ROUTED, OUTF32, X32>;
  if (const int rc = allow_dynamic_lds(reinterpret_cast<const void*>(fn), H::kLds); rc != BRT_OK) return rc;
  hipLaunchKernelGGL(fn, dim3(static_cast<unsigned>((blocks * a.tiles_n + kXcds - 1) / kXcds * kXcds)), dim3(kWaves * kWave), H::kLds, st, a);
  return check_launch("grouped_gemm_skinny_kernel");
}

template <int XR, int NT, int D, int ACT, bool X32>
int launch_of(GemmArgs& a, hipStream_t st) {
  const bool f32 = a.out_f32 != nullptr;
  if (a.tags != nullptr) return f32 ? launch<XR, NT, D, ACT, true, true, X32>(a, st) : launch<XR, NT, D, ACT, true, false, X32>(a, st);
  return f32 ? launch<XR, NT, D, ACT, false, true, X32>(a, st) : launch<XR, NT, D, ACT, false, false, X32>(a, st);
}

template <int XR, int NT, int D, bool X32 = false>
int launch_act(GemmArgs& a, int act, hipStream_t st) {
  if (act == BRT_ACT_GELU) return launch_of<XR, NT, D, BRT_ACT_GELU, X32>(a, st);
  if (act == BRT_ACT_RELU) return launch_of<XR, NT, D, BRT_ACT_RELU, X32>(a, st);
  return launch_of<XR, NT, D, BRT_ACT_NONE, X32>(a, st);
}

}  // namespace

// Where this kernel is taken, against the 160-row kernel.  Both were timed on 1 to 2000 rows per expert,
// 2 to 128 experts and 2 MB to 1 GB of weights (us, 160-row kernel -> this one); the rule gives up small gains
// rather than lose where the 160-row kernel is the faster one.
//   - Up to 28 rows per expert (one row block): while the weights are less than 0.3 GB (8 experts x 3 rows
//     3072 -> 768 43.7 -> 11.2, 32 x 6 rows 4096 -> 1024 62.9 -> 55.2, 1024 -> 4096 47.6 -> 46.5).  Beyond, the wide
//     tiles stream them at the memory's rate (32 x 24 rows 2560 -> 1920, 314 MB: 56.0 there, 60.3 here; 64 x 6 rows
//     1024 -> 4096, 536 MB: 86.8 and 90.7), except where they cannot: half of the CUs without a tile
//     (16 x 12 rows 6656 -> 1664 89.6 -> 64.5), a K whose rows lie multiples of 4 KB apart (64 x 16 rows
//     4096 -> 1024 120.8 -> 108.3, 32 x 20 rows 2048 -> 2560 80.9 -> 65.8) or experts of which many get no
//     row at all; up to 1 GB (32 x 8 rows 8192 -> 2048, 1.07 GB: 163 there, 226 here).
//   - Up to 64 rows: every block of rows streams the weights again (from the L2), which pays while the
//     160-row kernel has too few 160 x 256 tiles for the CUs: up to 72 of them, and up to 160 with less than
//     0.15 GB (16 x 64 rows 512 -> 2048 14.4 -> 10.1, 32 x 40 rows 768 -> 1024 17.2 -> 13.8, 16 x 60 rows
//     1024 -> 2560, 160 tiles, 21.5 -> 20.9; not 16 x 40 rows 3840 -> 1920, 236 MB).
//   - More: up to 96 tiles (8 x 120 rows 768 -> 3072 19.0 -> 15.6, 3072 -> 768 46.4 -> 21.0, 16 x 100 rows
//     768 -> 1536 18.6 -> 15.1; 112 tiles, 14 x 120 rows 1024 -> 2048: 22.3 there, 23.3 here; 144 tiles, 16 x 120
//     rows 1024 -> 2304: 22.7 and 30.5) of up to 32 experts (32 x 120 rows 2048 -> 512 35.1 -> 25.3),
//     and up to 160 with fewer experts than XCDs, some of which the 160-row kernel leaves idle (4 x 120 rows
//     2048 -> 8192 69.3 -> 41.9).
//     With 24 experts or more, up to 400 rows each, the contracting shapes that are dealt by expert, up to 100 tiles and 70 MB of
//     weights or 150 and 40: their rows and weights come to an L2 once, where the 160-row kernel's few tiles leave CUs idle and each walks
//     all of K (64 x 120 rows 2048 -> 256 37.1 -> 25.7, 1024 -> 256 22.0 -> 13.6, 48 x 204 rows 512 -> 128 17.7 -> 6.8, 24 x 216 rows
//     1920 -> 640 38.8 -> 36.5).  Of 110 drawn shapes that this takes from that kernel the mean is 1.79 times as fast, one is slower
//     (32 x 352 rows 1536 -> 384 32.5 and 34.3).  Not with fewer experts (16 x 280 rows 1280 -> 1280 30.5 and 40.5), more tiles
//     (128 x 224 rows 256 -> 256 15.3 and 17.4) or more weights (128 x 181 rows 896 -> 224, 51 MB, 27.9 and 34.4).
bool few_rows_by_weight(const GemmArgs& a) {
  const long used = std::min(a.E, a.P);
  const long tiles = wide_tiles(a);
  const double weight_bytes = 2.0 * used * a.N * a.K;
  if (a.P > 64 * used) {
    if (expanding_and_dealt(a)) return true;
    if (used >= 24 && a.P <= 400 * used && tiles <= 150 && weight_bytes <= (tiles <= 100 ? 7e7 : 4e7) && experts_stay_on_an_xcd(a)) return true;
    if (tiles <= 96) return used <= 32;
    return a.P <= 128 * used && tiles <= 160 && used < 8 && weight_bytes < 1.5e8;
  }
  if (tiles <= 72) return true;
  if (a.P <= 28 * used) {
    if (weight_bytes < 3e8) return true;
    return weight_bytes < 1e9 && (tiles <= 128 || a.K % 2048 == 0 || 2l * a.P <= 3 * used);
  }
  return tiles <= 160 && weight_bytes < 1.5e8;
}

// Besides, with any weight, few rows whose weight rows are no whole 128-byte lines: this kernel keeps the memory's rate there
// (64 x 4 rows 1432 -> 4680 146 us), the wide tiles, which walk the lines of 256 columns at a time, do not (181).  68 drawn shapes of
// 0.3 to 4.2 GB, 1 to 20 rows per expert: 0.85 of the wide tiles' time in the mean; with more rows, or more than 12 and a long K, the
// two are level or those win (64 x 15 rows 4848 -> 2032 241 us here, 234 there; 64 x 31 rows 5152 -> 680 100 and 93).  An expert with many of the
// rows reads its weights again for every 32 of them, and still skewed loads gain more than even ones, as the wide tiles then wait for
// that expert's: of 69 skewed loads of 33 drawn shapes, 1 to 20 rows on average and up to 1194 with one expert, 0.69 of their time in the mean and 0.94
// at worst (64 x 19 rows 2400 -> 1248 85 us and 94 with 368 of them on one expert, 32 x 16 rows 2040 -> 4992 156 and 182 with 492), of 171 even ones
// 0.91, the worst 1.07 (32 x 19 rows 3976 -> 6136 329 and 308).
bool skinny_gemm_applies(const GemmArgs& a) {
  const long used = std::min(a.E, a.P);
  return few_rows_by_weight(a) || (a.K % kBK != 0 && a.P <= (a.K < 4096 ? 20 : 12) * used);
}

namespace {
bool takes_64_rows(const GemmArgs& a) { return a.P > 32l * std::min(a.E, a.P) && narrow_tiles(a, 64) >= 192; }
}  // namespace

// Where fp32 rows are rounded by this kernel, of the shapes of up to 64 rows per expert whose bf16 rows it takes
// (few_rows_by_weight): where it is faster than the cast kernel and the bf16 form behind each other.  It saves a
// launch and a pass over the rows, but every column tile reads twice the bytes of the rows again, and fewer stages
// fit the LDS.  The line was drawn on 3757 shapes (1 to 64 rows per expert, 4 to 128 experts, K 256 to 8192, N 512
// to 8192, rows in order or gathered for one or two paths; both sides back to back in a graph; more rows lose: 32
// x 120 rows 2048 -> 512 39.5 us cast and GEMM, 48.9 here): 28 of the 2899 it takes are more than 2 % slower than
// cast and GEMM, the worst 6 % (128 x 28 rows 520 -> 1032 gathered 45.0 us cast, 47.7 here), and the mean is 11 %
// faster.  Of 900 other shapes drawn from those ranges, half of them with ragged loads, it takes 772: 16 are over
// 2 % slower (the worst 4 x 32 ragged rows 1792 -> 7168, 29.0 and 33.6), the mean is 13 % faster.  Not taken (us,
// cast and GEMM, this kernel):
//   - 64-row tiles with 10 MB of rows or more (64 x 64 rows 2048 -> 512 50.0 and 59.0), a K beyond 2048, 0.12 GB of
//     weights (4 x 64 rows 2048 -> 8192 36.0 and 37.4), or rows gathered for several paths, which the cast reads only
//     once, unless K is short (12 x 64 rows 768 -> 3072 for two paths 21.9 and 23.8);
//   - 32 x 32 tiles with a K beyond 2048, whose chain four stages do not cover (4 x 8 rows 4096 -> 1024 16.5 and 18.6),
//     except where the tiles reach most CUs (8 x 16 rows 4096 -> 1024 24.5 and 21.4, 12 x 8 rows 2560 -> 640 17.1 and 14.5);
//   - 32 x 64 tiles with more than 32 rows and a K beyond 2048 (12 x 64 rows 3072 -> 768 36.2 and 38.5), with 16 MB of
//     rows (128 x 28 rows 1536 -> 512 52.2 and 55.3), and a K from 2048 on whose few rows cost no time to cast beside 0.12 GB
//     of weights (64 x 3 rows 2048 -> 1024 55.7 and 57.1).
// cells: rows of x where they are gathered, 0 where they are not.
bool skinny_gemm_takes_f32(const GemmArgs& a, int cells) {
  const long used = std::min(a.E, a.P);
  const double row_bytes = 4.0 * a.P * a.K, weight_bytes = 2.0 * used * a.N * a.K;
  if (takes_64_rows(a))
    return a.K <= 2048 && row_bytes <= 1e7 && weight_bytes <= 1.2e8 && (cells == 0 || cells >= a.P || a.K <= 512);
  if (narrow_tiles(a, 32) <= 128)
    return a.K <= 2048 || (a.K <= 4096 && used * ((a.N + 63) / 64) >= 96 && (a.K <= 2560 || a.P >= 16 * used));
  if (a.P > 32 * used) return a.K <= 2048;
  return row_bytes <= 1.6e7 && (a.K < 2048 || a.P >= 16 * used || weight_bytes <= 1.2e8);
}

// Shape of the tile.
//   - 64 x 64 where experts have more than 32 rows and that makes a tile for most CUs (8 x 120 rows
//     768 -> 3072 15.7 us, 19.3 with 32 x 64): with a short K three stages and three workgroups on a CU
//     (16 x 64 rows 512 -> 2048 10.2 us, four stages 11.5), else four (8 x 120 rows 3072 -> 768 20.9, three 22.7).
//   - 32 x 32 where even 32 x 64 would leave half of the CUs without a tile (8 x 3 rows 3072 -> 768 11.2 us, 13.4),
//     and for a short K with so few rows that reading them twice as often costs nothing (32 x 6 rows
//     1024 -> 4096 46.2 us, 50.0).
//   - 32 x 64 otherwise (8 x 28 rows 4096 -> 1024 19.8 us, 32 x 32 22.4; 32 x 6 rows 4096 -> 1024 55.1 and 62.2).
int launch_skinny_gemm(GemmArgs& a, int act, hipStream_t st) {
  const double rows = static_cast<double>(a.P) / std::min(a.E, a.P), tiles32 = narrow_tiles(a, 32);
  const bool tall = takes_64_rows(a);
  if (a.x_f32) {
    // fp32 rows take twice the room, so 64 x 64 tiles have three stages, two workgroups on a CU (4 x 33 rows 1024 -> 4096
    // 11.8 us, two stages 16.5, cast and bf16 13.2; 8 x 40 rows 1024 -> 2048 12.0, 16.7 and 13.7), and two stages and three
    // workgroups where there are two tiles per CU and K is short (16 x 64 rows 640 -> 2560 22.7, three stages 23.3) or K is
    // hardly longer than the stages (384); 32 x 64 tiles have four (64 x 8 rows 512 -> 1024 16.7, 32 x 32 24.7, cast and bf16
    // 20.6; 8 x 3 rows 768 -> 3072 9.8, 12.9 and 11.7), and 32 x 32 are taken only where those leave half of the CUs without a
    // tile (8 x 28 rows 4096 -> 1024 22.1, 23.9 and 26.3).
    if (tall)
      return a.K <= 384 || (a.K <= 768 && narrow_tiles(a, 64) >= 512) ? launch_act<64, 2, 2, true>(a, act, st)
                                                                    : launch_act<64, 2, 3, true>(a, act, st);
    if (tiles32 <= 128) return launch_act<32, 1, 4, true>(a, act, st);
    return launch_act<32, 2, 4, true>(a, act, st);
  }
  if (tall) {
    if (a.K <= 1024) return launch_act<64, 2, 3>(a, act, st);
    return launch_act<64, 2, 4>(a, act, st);
  }
  if (tiles32 <= 112 || (tiles32 <= 160 && a.K <= 2048) || (rows <= 16 && a.K <= 1536)) return launch_act<32, 1, 6>(a, act, st);
  return launch_act<32, 2, 5>(a, act, st);
}

}  // namespace brt
