// Grouped expert GEMM, second kernel: 256 x 256 output tiles multiplied by two groups of
// wavefronts in ping-pong, for shapes that give an expert hundreds of rows and more (ragged
// task-MoE batches, top-2 routes with large capacities), where the matrix units and not the weight
// stream set the pace.
//
// Same contract as grouped_gemm.hip (out[rows of e] = act(x[rows of e] @ W_e^T + b_e), one launch,
// loads read on the device; reference: src/jit/compiler.cu:151-246).  What differs:
//
//   - A workgroup is 8 wavefronts, two per SIMD, each owning 128 x 64 outputs (32 accumulator tiles
//     of v_mfma_f32_16x16x32_bf16 = 128 registers, and the 24 fragments of a whole K-step of 64 in
//     96 more).  The wavefronts of a SIMD belong to two groups that run half a K-step apart: while
//     one group issues its 64 MFMAs (C phase), the other reads its fragments from LDS and requests
//     operands from memory (M phase); a workgroup barrier separates the phases.  The matrix pipe
//     of a SIMD therefore always has a wavefront that does nothing but multiply, and the memory
//     instructions of the other one never stand between two MFMAs.
//   - Operands go from global memory straight into LDS (buffer_load ... lds): no staging
//     registers.  The destination of such a load is M0 + 16 * lane, so the swizzle that keeps the
//     fragment reads free of bank conflicts is applied on the global side: the lane that fills
//     slot s of tile row r fetches chunk s ^ ((r >> 1) & 7) of that row.
//   - All 160 KB of LDS are operand stages: a ring of three K-steps of activation rows (32 KB
//     each) and a ring of two of weight rows.  Group 0 requests the activation rows two K-steps
//     ahead, into the slot both groups finished reading two phases earlier; group 1 requests the
//     weight rows two K-steps ahead into the slot it has just read itself (group 0 read the same
//     rows one phase earlier), once its own weight fragments are in registers.  Every request has
//     three to four phases to land, and each wavefront issues its 8 loads of a K-step in its M
//     phase, between fragment reads.  A K-step is 2 x 1024 clocks of MFMA per SIMD and measures
//     2150 to 2270, at the 1.5 to 1.8 GHz that the part sustains with them: it is the package's power that sets the time of a K-step
//     (1.3 to 1.45 us; with fewer clocks the clock rate falls), so what counts is its energy.  That of the 16 x 16 x 32 instruction is
//     lower than that of v_mfma_f32_32x32x16_bf16, which reads and writes every accumulator twice as often; both sum the products of
//     an output element to the same bits.  us, 32 x 32 x 16 and this: 8 x 4096 rows 2048 -> 8192 + GELU 906 and 876, 8192 -> 2048 776 and
//     752, 16 x 2048 rows 1024 -> 4096 + GELU 271 and 262, 4096 -> 1024 210 and 204, 64 x 400 rows 768 -> 3072 + GELU 161 and 155.
//     Four wavefronts of 128 x 128 outputs, the accumulators in the AGPRs (128 KB of fragment reads a K-step instead of 192, 2400 clocks at 1.75
//     GHz), need as much without an activation and 4 to 15 % more with GELU: nothing runs beside a wavefront's epilogue there.
//     The 64 KB of loads of a K-step alone take 0.62 us per CU when the rows are up to 8 KB apart and 1.08 us when they
//     are 16 KB apart (K = 8192: the 512 rows of a tile pair then lie in 128 regions of 64 KB,
//     more than a CU's address translation holds), so the load stream has to be fed in every
//     phase and must not wait for anything.
//   - Waits count the wavefront's own loads (s_waitcnt vmcnt(8): everything but the 8 loads of
//     this K-step has landed); the barrier that ends a phase publishes the data.
//   - Workgroups are numbered in patch order (see grouped_gemm.hip): 4 row blocks x 8 column tiles
//     of one expert on an XCD at a time, sharing both operands through that XCD's L2.
//   - Routed rows cost the K loop nothing: a wavefront keeps the byte offsets of the eight row groups
//     it loads in registers for any kind of row, so a gathered row (its cell's offset) and an
//     activation or weight row (row times pitch) are the same load.  The cells pass through the
//     first bytes of the stages once, before any operand lands there.
//   - A workgroup of the whole rounds walks two column tiles (or three or five) of its row block: the requests of the last K-steps
//     of a tile are the first ones of the next, and the images of the finished rows go through the one slot of the rings that is free.
//   - What the list of tiles holds beyond whole rounds over the CUs would keep a few of them busy for as long as a whole round, and the
//     experts' last row blocks, which hold few rows, for more than half as long (the weights of 256 columns come into one CU at
//     40 GB/s).  Where that is at most half a round it is cut into units of 256 rows x 64 columns: each wavefront loads its share of a
//     K-step and multiplies 32 rows (or 32 x 32 outputs of fewer rows) of a ring of four to eight K-steps, one barrier per K-step, the loads
//     between the MFMAs (in front of them a K-step took 0.65 us instead of 0.53).  Bound by the fills of LDS, 40 KB a
//     K-step at 64 bytes a clock.  32768 rows of 16 experts 4096 -> 1024 268 -> 229 us, 32 x 1000 rows 512 -> 1024 61 -> 50.
//   - The epilogue sends the tile out 32 rows at a time through each wavefront's own corner of
//     LDS (the stages are dead by then), full 128-byte rows per store.
#include <algorithm>
#include <type_traits>
#include <utility>

#include "common.hpp"
#include "grouped_gemm.hpp"
#include "rows.hpp"

namespace brt {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef const bf16x4 __attribute__((address_space(1)))* global_bf16x4;
typedef const __bf16 __attribute__((address_space(1)))* global_bf16;

constexpr int kWaves = 8;
constexpr int kMT = 8, kNT = 4;                       // 16 x 16 tiles per wavefront: 128 x 64
constexpr int kBM = 256, kBN = 256, kBK = 64;
constexpr int kRowB = kBK * 2;                        // bytes of one tile row in one stage: one cache line
constexpr int kTileB = kBM * kRowB;                   // one operand of one K-step: 32 KB
constexpr int kAStages = 3, kBStages = 2;
constexpr int kBBase = kAStages * kTileB;             // the weight ring follows the activation ring
constexpr int kLdsBytes = (kAStages + kBStages) * kTileB;  // 163840: all of a CU's LDS
constexpr int kSub = kBK / 32;                        // MFMA k-steps per stage
constexpr int kHead = 8;                              // MFMAs of a C phase issued ahead of the barrier
constexpr uint32_t kOutOfRange = 0xf0000000u;         // buffer offset past any extent, also with what a load adds: reads as zero
constexpr int kXcds = 8, kCusPerXcd = 32, kPatchRows = 4;
constexpr int kRoundBits = 8, kRound = kXcds * kCusPerXcd;  // tiles of a whole round
static_assert(kRound == 1 << kRoundBits);
// The end of the list that is cut into units (see the kernel).  It takes the CUs one round of units up to 64 tiles and two up to 128,
// against a round in which the tiles leave most CUs idle.  A unit of 256 rows takes 0.4 of a tile's time (4 x 1024 rows
// 4096 -> 1024, 256 units: 38 us against 90 us for the 64 tiles they are made of), one of up to 128 rows half of what its block
// takes as a tile.  Of lists of one to two and a half rounds (50 drawn ones; us, not cut and cut): up to 60 tiles 0.71 to 0.90 of the time (one 1.02),
// 61 to 76 tiles 0.80 to 1.01, 77 to 91 tiles 0.87 to 1.02 (4 x 1704 rows 1504 -> 3008 74 and 73), 92 to 104 tiles 0.95 to 1.05, 108 and more,
// which are left whole, 0.91 to 1.13 if they were cut (24 x 934 rows 3696 -> 984 198 and 221, 64 x 393 rows 2288 -> 736 125 and 135);
// where all of them are blocks of few rows 104 tiles 0.81 and 0.87 (60 x 265 rows 4152 -> 592 202 and 163), 128 of 128 rows 1.05
// (32 x 640 rows 6024 -> 928 307 and 322).  In a list of more than ten rounds the CUs are no longer in step, and nothing
// is left to gain (98 blocks 2048 -> 8192, 12.25 rounds: level).
constexpr int kFewRows = 128, kMostCut = 104, kMostCutOfFewRows = 116, kMostRounds = 10;
constexpr int kUnitCols = 64;
constexpr int kStreamed = 2 | 16;  // cache policy of a buffer store: nt sc1
struct ListEnd {
  int moved, cut;  // row blocks of few rows put behind the list, tiles cut in all
};
template <typename OverTn>
__host__ __device__ __forceinline__ ListEnd end_of_list(const GemmArgs& a, int tiles, int few, OverTn over_tn) {
  const int tn = a.tiles_n, rest = tiles & (kRound - 1);
  int moved = min(few, over_tn(rest + tn - 1));
  int cut = max(moved * tn, rest);
  const int most = moved * tn >= rest ? kMostCutOfFewRows : kMostCut;
  if (cut > most || tiles > kMostRounds * kRound || tiles + 3 * cut > a.grid - (a.row_tags_out != nullptr ? 1 : 0)) cut = 0;
  if (cut == 0) moved = 0;
  return {moved, cut};
}

__device__ __forceinline__ i32x4 make_rsrc(const void* p, size_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  i32x4 r;
  r[0] = static_cast<int>(a);
  r[1] = static_cast<int>((a >> 32) & 0xffff);
  r[2] = static_cast<int>(bytes > 0x7fffffffull ? 0x7fffffffull : bytes);
  r[3] = 0x00020000;
  return r;
}

// 16 bytes per lane from the buffer straight into LDS at lds_base + kAt + 16 * lane (wave-uniform lds_base in M0, one wait
// state between its write and the load); the instruction's offset kAt is added to the place in the buffer too.  Counts on vmcnt
// like any load; the compiler does not know it touches LDS, so every wait for such a load is written out below.
template <int kAt = 0>
__device__ __forceinline__ void load_to_lds(const i32x4& rsrc, uint32_t voffset, uint32_t soffset,
                                            uint32_t lds_base) {
  if constexpr (kAt == 0)
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "{m0}"(lds_base), "v"(voffset), "s"(rsrc), "s"(soffset)
                 : "memory");
  else  // M0 is what it was for the load before
    asm volatile("buffer_load_dwordx4 %1, %2, %3 offen offset:%4 lds"
                 :
                 : "{m0}"(lds_base), "v"(voffset), "s"(rsrc), "s"(soffset), "n"(kAt)
                 : "memory");
}
template <typename Fn, int... I>
__device__ __forceinline__ void for_each(Fn&& fn, std::integer_sequence<int, I...>) { (fn(std::integral_constant<int, I>{}), ...); }

// acc += w x, 16 x 16 x 32.  In place: as a builtin the instruction gets other registers for its result, and accumulators are moved.
// The compiler does not know its wait states then: mfma_wait_states() stands before anything else reads an accumulator.
__device__ __forceinline__ void multiply_add(f32x4& acc, const bf16x8& w, const bf16x8& x) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(w), "v"(x));
}
__device__ __forceinline__ void mfma_wait_states() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 15" : : : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// what is the same in all lanes, in scalar registers (the compiler cannot always tell)
__device__ __forceinline__ i32x4 in_scalars(i32x4 r) {
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = __builtin_amdgcn_readfirstlane(r[i]);
  return r;
}

__device__ __forceinline__ void stream_out(const u32x4& v, u32x4* p) {
  // (a store of more than 64 bits wants one wait state before its data registers are written again)
  asm volatile("global_store_dwordx4 %0, %1, off sc1 nt\n\ts_nop 0" : : "v"(p), "v"(v) : "memory");
}

__device__ __forceinline__ void wait_loads_all() { asm volatile("s_waitcnt vmcnt(0)" : : : "memory"); }
// everything but the 8 loads this wavefront issued in the current K-step has landed
__device__ __forceinline__ void wait_loads_but_8() { asm volatile("s_waitcnt vmcnt(8)" : : : "memory"); }
template <int N>
__device__ __forceinline__ void wait_loads_but() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory"); }
__device__ __forceinline__ void block_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <int ACT, bool ROUTED, bool OUTF32>
__global__ __launch_bounds__(kWaves * 64) void grouped_gemm_pingpong_kernel(GemmArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  // in the routed forms the cells behind the tile's rows pass through the first bytes of the stages, before any
  // load lands there
  int* const s_cell = reinterpret_cast<int*>(smem);  // 0-based cell of each row of the tile, -1 = empty slot

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Wavefronts w and w + 4 share a SIMD: wm is the half of the tile's rows a wavefront owns and
  // also its ping-pong group; wn is its 64 columns.
  const int wm = wave >> 2, wn = wave & 3;

  // ---- which tile ------------------------------------------------------------------------------
  // The list holds the tiles of the row blocks in patch order (grouped_gemm.hip).  What it holds beyond whole rounds over
  // the CUs is cut into units of 256 rows x 64 columns, four for a tile, if it is little: first the experts' last row blocks
  // of few rows, as far as needed (`moved` blocks, taken out of the list and put behind it), then the end of the list.
  // Every wavefront finds its tile by itself, the weight pointers fetched in the same round trip as the loads: no
  // exchange through LDS and no second trip stand before the first requests, and the K loop starts when the first K-step
  // has landed.  Against one wavefront that looks, LDS, a load of the pointer and a wait for two K-steps:
  // 16 x 2048 rows 1024 -> 4096 + GELU 278.8 -> 274.3 us (0.6 us a tile), 64 x 400 rows 768 -> 3072 174.1 -> 169.7, 8 x 4096 rows
  // 2048 -> 8192 907.9 -> 899.0; contracting GEMMs, whose tiles take four times as long, within 0.5 %.
  // (The 160-row kernel, which starts once per CU, lost 0.5 to 1 % by the same change.)
  // A lane looks at two experts: up to 128 of them take one round trip and one scan.
  const int xcd = blockIdx.x % kXcds, idx = blockIdx.x / kXcds;
  const int t = ((idx / kCusPerXcd) * kXcds + xcd) * kCusPerXcd + idx % kCusPerXcd;
  const int tn = a.tiles_n;
  struct Two {
    int m[2], many[2], few[2];  // rows; row blocks of more than kFewRows rows, and of fewer (one at most)
    int incl_m, incl_b;         // rows and blocks up to this lane's experts and with them (blocks of few rows in the low byte)
    uint64_t w[2];
  };
  auto read_two = [&](int base) {
    Two v;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int el = base + 2 * lane + i, at = min(el, a.E - 1);
      const int given = a.loads[at];
      v.w[i] = reinterpret_cast<uint64_t>(a.w[at]);
      v.m[i] = el < a.E ? given : 0;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int over = v.m[i] & (kBM - 1);
      v.many[i] = (v.m[i] >> 8) + (over > kFewRows ? 1 : 0);
      v.few[i] = over > 0 && over <= kFewRows ? 1 : 0;
    }
    v.incl_b = wave_inclusive_scan((v.many[0] + v.many[1]) << 8 | (v.few[0] + v.few[1]));
    v.incl_m = wave_inclusive_scan(v.m[0] + v.m[1]);
    return v;
  };
  auto over = [](int n, int d, uint32_t inverse) {  // n / d
    const int q = static_cast<int>(__umulhi(static_cast<uint32_t>(n), inverse));
    return n - q * d >= d ? q + 1 : q;
  };
  auto over_tn = [&](int n) { return over(n, tn, a.tiles_n_inverse); };
  auto over_walk = [&](int n) { return over(n, a.walk, a.walk_inverse); };
  Two two = read_two(0);
  const int sums = read_lane(two.incl_b, kWave - 1);
  int many = sums >> 8, few = sums & 255;
  for (int base = 2 * kWave; base < a.E; base += 2 * kWave) {
    const int more = read_lane(read_two(base).incl_b, kWave - 1);
    many += more >> 8, few += more & 255;
  }
  const int tiles = (many + few) * tn;
  const auto [moved, cut] = end_of_list(a, tiles, few, over_tn);
  const int listed = tiles - moved * tn, whole = tiles - cut;
  // Whole rounds over the CUs of `walk` tiles each come first, one workgroup for the column tiles of a row block.
  const int walkers = a.walk > 1 ? over_walk(whole >> kRoundBits) << kRoundBits : 0, walked = walkers * a.walk;
  const int used = walkers + (whole - walked) + 4 * cut;
  if (t >= used) {
    // Surplus workgroups clear the tags of the rows no path owns, 256 of them a step.  The grid holds P / 256 + E row blocks
    // (rounded up) per column tile, the experts use at most (total + 255 E) / 256, and the cut leaves at least one.
    if (ROUTED && a.row_tags_out != nullptr && tid < kBM) {
      long total = 0;
      for (int base = 0; base < a.E; base += 2 * kWave) total += read_lane(read_two(base).incl_m, kWave - 1);
      for (long r = total + static_cast<long>(t - used) * kBM + tid; r < a.P; r += static_cast<long>(gridDim.x - used) * kBM) a.row_tags_out[r] = 0;
    }
    return;
  }
  const int at = t < walkers ? t * a.walk : walked + (t - walkers);  // in the list, a unit counted as one
  const bool narrow = at >= whole;
  const int tile = narrow ? whole + ((at - whole) >> 2) : at;
  int left = t < walkers ? a.walk : 1;  // tiles of this workgroup, the one at hand included
  const bool apart = tile >= listed;  // of a moved block
  const int place = apart ? tile - listed : tile;
  int e = 0, row0 = 0, rows = 0, seat0 = 0, n0 = 0;
  const __bf16* w_e = nullptr;
  for (int base = 0, carry_many = 0, carry_few = 0, carry_m = 0;;) {
    const int few_own = two.few[0] + two.few[1], many_own = two.many[0] + two.many[1];
    const int few_with = carry_few + (two.incl_b & 255), few_before = few_with - few_own;
    const int many_with = carry_many + (two.incl_b >> 8);
    const int first = apart ? min(few_before, moved) : many_with - many_own + max(few_before - moved, 0);
    const int last = apart ? min(few_with, moved) : many_with + max(few_with - moved, 0);
    const unsigned long long hit = __ballot(place >= first * tn && place < last * tn);
    if (hit != 0) {
      const int src = __builtin_ctzll(hit);
      int local = place - read_lane(first, src) * tn;  // among the tiles of the lane's two experts
      const int before = read_lane(few_before, src), few0 = read_lane(two.few[0], src), few1 = read_lane(two.few[1], src);
      const int many0 = read_lane(two.many[0], src), many1 = read_lane(two.many[1], src);
      const int m0 = read_lane(two.m[0], src), m1 = read_lane(two.m[1], src);
      // blocks of the first of them that are looked for
      const int moved0 = few0 != 0 && before < moved ? 1 : 0, moved1 = few1 != 0 && before + few0 < moved ? 1 : 0;
      const int blocks0 = apart ? moved0 : many0 + few0 - moved0;
      const bool second = local >= blocks0 * tn;
      if (second) local -= blocks0 * tn;
      const int m = second ? m1 : m0;
      int block, col;
      if (apart) {
        block = second ? many1 : many0;
        col = local;
      } else {
        const int blocks = second ? many1 + few1 - moved1 : blocks0;
        const int g = min(over_tn(local) / kPatchRows, blocks / kPatchRows);
        // of a patch the first a.walk column tiles of its row blocks, one row block after the other, then the next ones (a.walk divides tn)
        const int r = local - g * kPatchRows * tn, wide = min(blocks - g * kPatchRows, kPatchRows);
        const int run = a.walk > 1 ? over_walk(r) : r;
        const int runs = wide == 4 ? run >> 2 : wide == 3 ? static_cast<int>(__umulhi(static_cast<uint32_t>(run), 0x55555556u)) : wide == 2 ? run >> 1 : run;
        block = g * kPatchRows + run - runs * wide;
        col = runs * a.walk + r - run * a.walk;
      }
      const uint64_t wp = second ? two.w[1] : two.w[0];
      e = base + 2 * src + (second ? 1 : 0);
      seat0 = block * kBM;
      row0 = carry_m + read_lane(two.incl_m, src) - m1 - (second ? 0 : m0) + seat0;
      rows = min(min(kBM, m - seat0), a.P - row0);
      n0 = col * kBN;
      w_e = reinterpret_cast<const __bf16*>(static_cast<uint64_t>(static_cast<uint32_t>(read_lane(static_cast<int>(wp), src))) |
                                            static_cast<uint64_t>(static_cast<uint32_t>(read_lane(static_cast<int>(wp >> 32), src))) << 32);
      break;
    }
    carry_many += read_lane(two.incl_b, kWave - 1) >> 8;
    carry_few += read_lane(two.incl_b, kWave - 1) & 255;
    carry_m += read_lane(two.incl_m, kWave - 1);
    base += 2 * kWave;
    if (base >= a.E) return;  // (no tile of the list is here)
    two = read_two(base);
  }
  if (narrow) {
    n0 += ((at - whole) & 3) * kUnitCols;
    if (n0 >= a.N) return;
  }
  const int K = a.K;
  const int k_tiles = __builtin_amdgcn_readfirstlane((K + kBK - 1) / kBK);
  // A last K-step that K does not fill: before it is requested, and nothing after it is, the lanes whose chunk of 8 elements
  // lies behind K are turned to an offset past any extent, so they fill LDS with zeros.  (K is a multiple of 8.)  The K loop
  // pays one scalar comparison for it: 16 x 2048 rows 1024 -> 4096 282.8 us without it, 281.5 with it.
  const int part = K % kBK != 0 ? k_tiles - 1 : -1;  // that K-step
  auto cut_chunk = [&](uint32_t& offset, int group) {  // of this lane's load of a row group
    int l = lane;
    asm volatile("" : "+v"(l));  // (else its comparisons are kept in registers all through the K loop)
    if (((l & 7) ^ ((group * 4 + (l >> 4)) & 7)) * 8 >= K % kBK) offset = kOutOfRange;
  };
  if constexpr (ROUTED) {  // one word per row, all of them in one round trip
    if (tid < kBM) {
      const int cell = tid < rows ? routed_cell(a, e, row0 + tid, seat0 + tid) : -1;
      s_cell[tid] = cell;
      // side output for a combine that runs later: written once per row block
      if (a.row_tags_out != nullptr && n0 == 0 && tid < rows) a.row_tags_out[static_cast<size_t>(row0) + tid] = cell + 1;
    }
    __syncthreads();
  }

  // MFMA operand: this lane feeds row lane % 16, chunk lane / 16 (of 8 elements) of a 16 x 32 block; chunk
  // ks * 4 + lane / 16 of a stage's row sits in slot chunk ^ ((row >> 1) & 7)
  const int frag_row = lane & 15, frag_k = lane >> 4;
  const int swz = (frag_row >> 1) & 7;
  auto frag_off = [&](int ks) { return ((ks * 4 + frag_k) ^ swz) << 4; };
  const bool gather = ROUTED && a.gather != 0;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem)));

  // ---- epilogue: bias + activation, bf16, 32 rows at a time through this wavefront's image -----
  // transposed accumulator: element r of tile (i, j) is output row 16 i + lane % 16, column (of the
  // wavefront's) 16 j + 4 * (lane / 16) + r, i.e. a lane holds 4 consecutive columns (8 bytes) of its row.
  // Rows and columns that are not there are left to the bounds of the buffer that is stored to, and without a bias nothing is added
  // (a sum of products that starts at +0 is never -0).  With a branch for each row and a zero added, and so, us: 4 x 8000 rows 256 -> 1024 + GELU 31.5
  // and 30.3, 16 x 2048 rows 1024 -> 4096 + GELU 252 and 247, 8 x 4096 rows 8192 -> 2048 746 and 736.
  auto epilogue = [&](auto& acc, int first_row, int mine, int col_w, uint32_t images, auto with_bias) {
    constexpr int MT = sizeof(acc) / sizeof(acc[0]), NT = sizeof(acc[0]) / sizeof(acc[0][0]);
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane), "+s"(images));  // (else what follows from it is kept in registers all through the K loops of a walk)
    const int frag_row = lane & 15, frag_k = lane >> 4;
    const int row_w = row0 + first_row;
    constexpr int kOutB = OUTF32 ? 4 : 2;                 // bytes of one output element
    constexpr int kChunk = 16 / kOutB;                    // elements of one 16-byte store
    constexpr int kCols = OUTF32 ? 32 : NT * 16;          // columns of an image
    constexpr int kChunksPerRow = kCols / kChunk;
    constexpr int kImageRow = kCols * kOutB, kImageB = 32 * kImageRow;
    static_assert(kWaves * kImageB <= kTileB, "the output images must fit one slot");
    char* const image = smem + images + wave * kImageB;
    // the chunks of an image row are swizzled like those of the stages
    auto slot = [](int row, int chunk) { return (chunk ^ (kChunksPerRow == 4 ? (row >> 2) & 3 : (row >> 1) & 7)) * 16; };
    constexpr int kRowsPerPass = kWave / kChunksPerRow;
    // the bias of this lane's columns, all loads in one round trip
    constexpr bool kBias = decltype(with_bias)::value;
    bf16x4 bv[NT];
    if constexpr (kBias) {
      const global_bf16 bias = (global_bf16)(a.bias[e]);
  #pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int col = col_w + j * 16 + 4 * frag_k;
        bv[j] = bf16x4{};
        if (col < a.N) bv[j] = *(global_bf16x4)(bias + col);
      }
    }
    const bool scatter = ROUTED && a.scatter != 0;
    char* const out_b = OUTF32 ? reinterpret_cast<char*>(a.out_f32) : reinterpret_cast<char*>(a.out);
    const uint32_t row_b = static_cast<uint32_t>(a.N) * kOutB;
    const __amdgpu_buffer_rsrc_t to_rows = __builtin_amdgcn_make_buffer_rsrc(
        out_b + static_cast<size_t>(row_w) * row_b, 0, static_cast<int>(max(mine, 0) * row_b), 0x00020000);
  #pragma unroll
    for (int i = 0; i < MT / 2; ++i) {
      if (i * 32 >= mine) break;  // wave-uniform
      // scattered rows: lane r of the pass holds the cell of row r (read again: LDS held operands)
      int cell = -1;
      if (scatter && lane < min(32, mine - i * 32)) {
        const int r = row_w + i * 32 + lane;
        cell = routed_cell(a, e, r, r - row0 + seat0);
      }
  #pragma unroll
      for (int j0 = 0; j0 < NT; j0 += kCols / 16) {
  #pragma unroll
        for (int ii = 0; ii < 2; ++ii) {
  #pragma unroll
          for (int j = j0; j < j0 + kCols / 16; ++j) {
            float v[4];
  #pragma unroll
            for (int q = 0; q < 4; ++q) {
              const float sum = acc[2 * i + ii][j][q];
              v[q] = apply_act<ACT>(kBias ? sum + static_cast<float>(bv[j][q]) : sum);
            }
            const int row = ii * 16 + frag_row, at = (16 * (j - j0) + 4 * frag_k) * kOutB;  // in the image
            char* const to = image + row * kImageRow + slot(row, at / 16) + at % 16;
            if constexpr (OUTF32) {
              *reinterpret_cast<f32x4*>(to) = f32x4{v[0] + 0.0f, v[1] + 0.0f, v[2] + 0.0f, v[3] + 0.0f};  // -0 -> +0, as a combine would
            } else {
              *reinterpret_cast<bf16x4*>(to) = bf16x4{static_cast<__bf16>(v[0]), static_cast<__bf16>(v[1]),
                                                      static_cast<__bf16>(v[2]), static_cast<__bf16>(v[3])};
            }
          }
        }
        wave_fence();
        const int c = lane % kChunksPerRow, col = col_w + j0 * 16 + c * kChunk;
        constexpr int kPasses = 32 / kRowsPerPass;
        u32x4 held[kPasses];
  #pragma unroll
        for (int p = 0; p < kPasses; ++p) {
          const int row = p * kRowsPerPass + lane / kChunksPerRow;
          held[p] = *reinterpret_cast<const u32x4*>(image + row * kImageRow + slot(row, c));
        }
        if (scatter) {
  #pragma unroll
          for (int p = 0; p < kPasses; ++p) {
            const int to_row = __shfl(cell, p * kRowsPerPass + lane / kChunksPerRow, kWave);
            if (to_row < 0 || col >= a.N) continue;
            if constexpr (!OUTF32) {  // the combine this store stands for adds the row to zero: -0 becomes +0
  #pragma unroll
              for (int w = 0; w < 4; ++w) held[p][w] = plus_zero<BRT_BF16>(held[p][w]);
            }
            u32x4* const to = reinterpret_cast<u32x4*>(out_b + static_cast<size_t>(to_row) * row_b + col * kOutB);
            if (a.plain_out) *to = held[p];
            else stream_out(held[p], to);
          }
        } else {
          uint32_t at = col < a.N ? static_cast<uint32_t>(i * 32 + lane / kChunksPerRow) * row_b + col * kOutB : kOutOfRange;
          auto store = [&](auto policy) {
  #pragma unroll
            for (int p = 0; p < kPasses; ++p, at += kRowsPerPass * row_b)
              __builtin_amdgcn_raw_buffer_store_b128(held[p], to_rows, at, 0, decltype(policy)::value);
          };
          if (a.plain_out) store(std::integral_constant<int, 0>{});
          else store(std::integral_constant<int, kStreamed>{});
        }
        wave_fence();
      }
    }
  };

  // ---- a unit of the end of the list: `rows` rows, 64 columns from n0 on ---------------------------
  if (narrow) {
    const i32x4 res_x = in_scalars(gather ? make_rsrc(a.x, static_cast<size_t>(a.T) * K * 2)
                                          : make_rsrc(a.x + static_cast<size_t>(row0) * K, static_cast<size_t>(a.P - row0) * K * 2));
    const i32x4 res_u = in_scalars(make_rsrc(w_e + static_cast<size_t>(n0) * K, static_cast<size_t>(a.N - n0) * K * 2));
    auto unit = [&](auto rows_tag) {
      constexpr int UR = decltype(rows_tag)::value;         // rows of the unit
      constexpr int kXw = UR / 64, kL = kXw + 1;            // row groups of x a wavefront loads, loads of a K-step
      constexpr int UMT = 2, UNT = UR == 256 ? 4 : 2;       // 16 x 16 tiles of a wavefront: 32 rows, all columns or half of them
      constexpr int kStage = (UR + kUnitCols) * kRowB;
      constexpr int D = UR == 256 ? 4 : UR == 128 ? 6 : 8;  // K-steps in flight and in LDS
      static_assert(D * kStage <= kLdsBytes, "the ring must fit");
      uint32_t off[kL];
#pragma unroll
      for (int i = 0; i < kL; ++i) {
        const int row = (i == 0 ? wave : wave * kXw + i - 1) * 8 + (lane >> 3);
        const uint32_t chunk = (lane & 7) ^ ((row >> 1) & 7);
        int at = row;
        bool there = row < (i == 0 ? a.N - n0 : rows);
        if constexpr (ROUTED) {
          if (gather && i > 0) {
            at = s_cell[row];
            there = at >= 0;
          }
        }
        off[i] = there ? (static_cast<uint32_t>(at) * K + chunk * 8) * 2 : kOutOfRange;
      }
      if constexpr (ROUTED) __syncthreads();  // everyone has read the cells
      auto fetch = [&](int s, uint32_t stage, int i) {
        load_to_lds(i == 0 ? res_u : res_x, off[i], s * kRowB, lds0 + stage + (i == 0 ? UR / 8 + wave : wave * kXw + i - 1) * 1024);
      };
      const int tile_x = UNT == 4 ? wave : wave >> 1, tile_w = UNT == 4 ? 0 : wave & 1;
      const int first_row = tile_x * 32, mine = __builtin_amdgcn_readfirstlane(max(min(rows - first_row, 32), 0));
      f32x4 acc[UMT][UNT];
#pragma unroll
      for (int i = 0; i < UMT; ++i)
#pragma unroll
        for (int j = 0; j < UNT; ++j) acc[i][j] = f32x4{};
      struct Frags {
        bf16x8 w[kSub][UNT], x[kSub][UMT];
      };
      const char* const from_x = smem + (first_row + frag_row) * kRowB;
      const char* const from_w = smem + (UR + tile_w * 32 + frag_row) * kRowB;
      constexpr int kReads = UMT + UNT;  // of a k-step
      auto read_frag = [&](Frags& f, uint32_t stage, int q) {
        const int ks = q / kReads, of = q % kReads;
        if (of < UNT) f.w[ks][of] = *reinterpret_cast<const bf16x8*>(from_w + stage + frag_off(ks) + of * 16 * kRowB);
        else f.x[ks][of - UNT] = *reinterpret_cast<const bf16x8*>(from_x + stage + frag_off(ks) + (of - UNT) * 16 * kRowB);
      };
      auto cut_off = [&] {
#pragma unroll
        for (int i = 0; i < kL; ++i) cut_chunk(off[i], i == 0 ? wave : wave * kXw + i - 1);
      };
      const int primed = min(D, k_tiles);
      for (int s = 0; s < primed; ++s) {
        if (s == part) cut_off();
#pragma unroll
        for (int i = 0; i < kL; ++i) fetch(s, s * kStage, i);
      }
      // all but the last `younger` K-steps requested have landed
      auto landed = [&](int younger) {
        if (younger >= D - 1) wait_loads_but<(D - 1) * kL>();
        else if (younger == D - 2) wait_loads_but<(D - 2) * kL>();
        else if (D > 4 && younger == D - 3) wait_loads_but<(D > 4 ? D - 3 : 1) * kL>();
        else if (D > 5 && younger == D - 4) wait_loads_but<(D > 5 ? D - 4 : 1) * kL>();
        else if (D > 6 && younger == D - 5) wait_loads_but<(D > 6 ? D - 5 : 1) * kL>();
        else if (D > 7 && younger == D - 6) wait_loads_but<(D > 7 ? D - 6 : 1) * kL>();
        else if (younger == 1) wait_loads_but<kL>();
        else wait_loads_all();
      };
      landed(primed - 1);
      block_barrier();
      uint32_t stage = 0;
      auto step = [&](const Frags& cur, Frags& next, int s, auto multiply, auto fills) {
        constexpr bool kMultiply = decltype(multiply)::value, kFills = decltype(fills)::value;
        const uint32_t ahead = stage == (D - 1) * kStage ? 0 : stage + kStage;
        if (s + D == part) cut_off();
        if constexpr (kFills) wait_loads_but<(D - 2) * kL>();
        else landed(min(s + D - 1, k_tiles - 1) - (s + 1));
        block_barrier();
        if (!kFills && s + D < k_tiles) {
#pragma unroll
          for (int i = 0; i < kL; ++i) fetch(s + D, stage, i);
        }
        // the MFMAs of the K-step, and evenly behind them the reads for the next one and the requests
        constexpr int kMfmas = kSub * UMT * UNT;
#pragma unroll
        for (int n = 0; n < kMfmas; ++n) {
          if constexpr (kMultiply) {
            const int ks = n / (UMT * UNT), i = n / UNT % UMT, j = n % UNT;
            multiply_add(acc[i][j], cur.w[ks][j], cur.x[ks][i]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = n * kSub * kReads / kMfmas; q < (n + 1) * kSub * kReads / kMfmas; ++q) read_frag(next, ahead, q);
          }
          if constexpr (kFills) {
#pragma unroll
            for (int i = n * kL / kMfmas; i < (n + 1) * kL / kMfmas; ++i) fetch(s + D, stage, i);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (kMultiply) wait_lds();
        stage = ahead;
      };
      auto loop = [&](auto multiply) {
        Frags f0, f1;
        if constexpr (decltype(multiply)::value) {
#pragma unroll
          for (int q = 0; q < kSub * kReads; ++q) read_frag(f0, 0, q);
          wait_lds();
        }
        int s = 0;
        for (; s + 1 + D < k_tiles; s += 2) {
          step(f0, f1, s, multiply, std::true_type{});
          step(f1, f0, s + 1, multiply, std::true_type{});
        }
        for (; s < k_tiles; s += 2) {
          step(f0, f1, s, multiply, std::false_type{});
          if (s + 1 < k_tiles) step(f1, f0, s + 1, multiply, std::false_type{});
        }
      };
      if (mine > 0) {
        loop(std::true_type{});
        mfma_wait_states();
        if (a.bias != nullptr) epilogue(acc, first_row, mine, n0 + tile_w * 32, 0, std::true_type{});
        else epilogue(acc, first_row, mine, n0 + tile_w * 32, 0, std::false_type{});
      } else {
        loop(std::false_type{});
      }
    };
    if (rows <= 64) unit(std::integral_constant<int, 64>{});
    else if (rows <= 128) unit(std::integral_constant<int, 128>{});
    else unit(std::integral_constant<int, 256>{});
    return;
  }

  // ---- global -> LDS ---------------------------------------------------------------------------
  // A load fills one row group: 8 tile rows, a whole 128-byte line of each.  Group 0 loads the
  // activation rows, group 1 the weight rows, wavefront wn row groups 8 wn + i (i = 0..7).  Lane l lands at slot
  // l & 7 of row l >> 3 of the group and fetches chunk (l & 7) ^ ((row >> 1) & 7) of that row.  A row
  // that does not exist (past the expert's last row, past N) gets an offset past any extent: zeros,
  // no memory request.
  // Every wavefront keeps the eight offsets of its rows in registers (the K-step alone goes into
  // the scalar offset).  Gathered rows need that -- the cells of a row group are anywhere in x --
  // and it takes the bounds check out of the loop for the others.
  // An M phase is as long as its instructions take to issue, so the eight requests are eight instructions and two writes of M0: four
  // loads share one value, the instruction's own offset, 1 KB apart, moves them in LDS, and the registers hold the place in the
  // buffer less that offset, in a buffer that starts kBack bytes early.  When nothing more is to be requested the extent becomes
  // kBack, which no offset is below, and the scalar offset 0: whether a request is in range must not hang on a scalar offset that is more
  // than the extent (by the documents a raw buffer's bound is the extent less the scalar offset).  (With M0 computed and written for each load and a branch around it, against this, of the time that the kernel took with neither and
  // 32 x 32 x 16 MFMAs: 8192 -> 2048 0.983 and 0.952, 2048 -> 8192 0.964 and 0.932, ragged loads 8192 -> 2048 1.01 and 0.97.)
  constexpr uint32_t kBack = 3 * 1024;
  static_assert(kBack >= kRowB, "the scalar offsets of the two last, empty K-steps are 0 and kRowB");
  auto start_early = [](i32x4 r) {
    const uint64_t at = (static_cast<uint64_t>(static_cast<uint32_t>(r[1])) << 32 | static_cast<uint32_t>(r[0])) - kBack;
    r[0] = static_cast<int>(at), r[1] = static_cast<int>(at >> 32) & 0xffff;
    r[2] = static_cast<int>(static_cast<uint32_t>(r[2]) + kBack);
    return r;
  };
  i32x4 res = in_scalars(start_early(wm == 0
      ? (gather ? make_rsrc(a.x, static_cast<size_t>(a.T) * K * 2)
                : make_rsrc(a.x + static_cast<size_t>(row0) * K, static_cast<size_t>(a.P - row0) * K * 2))
      : make_rsrc(w_e + static_cast<size_t>(n0) * K, static_cast<size_t>(a.N - n0) * K * 2)));
  const int cols = a.N - n0;  // weight rows that exist from n0 on
  uint32_t off[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = (wn * 8 + i) * 8 + (lane >> 3);
    const uint32_t chunk = (lane & 7) ^ ((row >> 1) & 7);
    int at = row;
    bool there = row < (wm == 0 ? rows : cols);
    if constexpr (ROUTED) {
      if (gather && wm == 0) {
        at = s_cell[row];
        there = at >= 0;
      }
    }
    off[i] = there ? (static_cast<uint32_t>(at) * K + chunk * 8) * 2 + kBack - (i & 3) * 1024 : kOutOfRange;
  }
  if constexpr (ROUTED) __syncthreads();  // everyone has read the cells; the loads may overwrite them
  const uint32_t lds_rows = lds0 + (wm == 0 ? 0 : kBBase) + wn * 8 * 1024;
  auto load = [&](uint32_t from, uint32_t slot, auto i) {
    load_to_lds<(i & 3) * 1024>(res, off[i], from, lds_rows + slot + (i & 4) * 1024);
  };

  // ---- fragments -------------------------------------------------------------------------------
  // The row tiles that hold rows are shared evenly by the two groups, group 0 taking the first `half`
  // rows: with 128 rows or fewer in one group the phases of a K-step would run one after the other.
  // (Halves fixed at 128 rows: the ragged FFN of 128 experts, 108 of its 201 row blocks part-filled,
  // 2556 -> 2532 us; top-2 over 16384 cells of 32 skewed experts 390 -> 387 us; two runs of one side
  // differ by half of that.)
  const int half = __builtin_amdgcn_readfirstlane(((rows + 63) >> 6) << 5);
  const int first_row = wm * half;  // of this wavefront, inside the tile
  const int frag_x = (first_row + frag_row) * kRowB;
  const int frag_w = kBBase + (wn * kNT * 16 + frag_row) * kRowB;

  f32x4 acc[kMT][kNT];
  bf16x8 fw[kSub][kNT], fx[kSub][kMT];
  const int mine = min(rows - first_row, half);  // rows of this wavefront
  // pairs of its row tiles that hold rows (wave-uniform)
  const int pairs = __builtin_amdgcn_readfirstlane(max((mine + 31) >> 5, 0));

  // Before the request of K-step `turn` some lanes' offsets change: those of the chunks behind K, or, where a walk goes on to a last
  // column tile of fewer than 256 columns (K is whole there), those of the weight rows that it does not have.
  auto cut_off = [&] {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (part >= 0) {
        cut_chunk(off[i], wn * 8 + i);
      } else if (wm == 1) {
        int l = lane;
        asm volatile("" : "+v"(l));
        if ((wn * 8 + i) * 8 + (l >> 3) >= a.N % kBN) off[i] = kOutOfRange;
      }
    }
  };
  // prologue: K-steps 0 and 1 (both whole: K >= 128)
  using Eight = std::make_integer_sequence<int, 8>;
  for_each([&](auto i) { load(0, 0, i); }, Eight{});
  for_each([&](auto i) { load(kRowB, kTileB, i); }, Eight{});
  wait_loads_but_8();  // K-step 0
  block_barrier();
  // The K-steps of a walk's tiles follow one another in the rings: the slots of the K-step being read and of the one being
  // requested, where the latter starts in its rows, and what takes it from the end of a tile's K to the start of the next tile's.
  uint32_t a_cur = 0, a_load = 2 * kTileB, b_cur = 0, from = 2 * kRowB;
  const uint32_t turn_back = (wm == 0 ? 0 : static_cast<uint32_t>(kBN) * K * 2) - static_cast<uint32_t>(k_tiles) * kRowB;
  const bool narrow_last = a.N % kBN != 0;
  // The K loop, for a wavefront whose first NI row tiles hold rows.  A ragged expert's last row
  // block reads no fragments and issues no MFMAs for the other row tiles, so a block of few rows
  // runs at the pace of its weight stream instead of that of 256 rows of matrix work.  The
  // wavefronts of a workgroup may run different instances: the barriers and the requests are the same in all.
  auto k_loop = [&](auto ni_tag) {
    constexpr int NI = decltype(ni_tag)::value;
    const int turn = left == 2 && narrow_last && n0 + 2 * kBN > a.N ? k_tiles : part;
    for (int kt = 0; kt < k_tiles; ++kt) {
      if (kt + 2 == turn) cut_off();
      if (kt + 2 == k_tiles) {
        from = left == 1 ? 0 : from + turn_back;
        if (left == 1) res[2] = kBack;
      }
      const char* const pa = smem + a_cur + frag_x;
      const char* const pb = smem + b_cur + frag_w;
      // ---- M phase: fragments of K-step kt into registers, requests for K-step kt + 2.  Group 0's activation rows go into the slot that
      // held K-step kt - 1: both groups have read it.  Group 1's weight rows go into the slot it is reading: group 0 read these rows a
      // phase ago, and this wavefront's own weight fragments are in registers after the wait.
      if constexpr (NI > 0) {
#pragma unroll
        for (int ks = 0; ks < kSub; ++ks)
#pragma unroll
          for (int j = 0; j < kNT; ++j) fw[ks][j] = *reinterpret_cast<const bf16x8*>(pb + frag_off(ks) + j * 16 * kRowB);
      }
      const uint32_t slot = wm == 0 ? a_load : b_cur;
      if (wm == 1) wait_lds();
      __builtin_amdgcn_sched_barrier(0);
      for_each(
          [&](auto i) {
            if constexpr (NI > 0) {
#pragma unroll
              for (int ks = 0; ks < kSub; ++ks)
                if (i < NI) fx[ks][i] = *reinterpret_cast<const bf16x8*>(pa + frag_off(ks) + i * 16 * kRowB);
            }
            load(from, slot, i);
          },
          Eight{});
      wait_lds();
      if (wm == 1) wait_loads_but_8();  // the weight rows of K-step kt + 1 have landed (group 0 reads them after this barrier)
      // MFMAs [first, last) of the K-step's 8 x NI, in (ks, i, j) order
      auto multiply = [&](auto first_tag, auto last_tag) {
        constexpr int kFirst = decltype(first_tag)::value, kLast = decltype(last_tag)::value;
#pragma unroll
        for (int ks = 0; ks < kSub; ++ks)
#pragma unroll
          for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < kNT; ++j) {
              const int n = (ks * NI + i) * kNT + j;
              if (n >= kFirst && n < kLast)
                multiply_add(acc[i][j], fw[ks][j], fx[ks][i]);
            }
      };
      // ---- C phase: nothing but the MFMAs of the K-step.  The first kHead of them are issued
      // before the barrier: they queue up behind the other group's last MFMAs and keep the matrix
      // pipe fed while the barrier lets both groups through (2.5 % on every shape measured; with twice
      // as many the group reaches the barrier too late for the other one's M phase).
      __builtin_amdgcn_sched_barrier(0);
      multiply(std::integral_constant<int, 0>{}, std::integral_constant<int, kHead>{});
      __builtin_amdgcn_sched_barrier(0);
      block_barrier();
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(1);
      multiply(std::integral_constant<int, kHead>{}, std::integral_constant<int, kSub * kMT * kNT>{});
      __builtin_amdgcn_s_setprio(0);
      __builtin_amdgcn_sched_barrier(0);
      if (wm == 0) wait_loads_but_8();  // the activation rows of K-step kt + 1 have landed
      // (group 1 goes from its last C phase straight into the epilogue)
      if (wm == 0 || kt + 1 < k_tiles) block_barrier();
      a_cur = a_cur == 2 * kTileB ? 0 : a_cur + kTileB;
      a_load = a_load == 2 * kTileB ? 0 : a_load + kTileB;
      b_cur ^= kTileB;
      from += kRowB;
    }
    if constexpr (NI > 0) mfma_wait_states();  // in here: where the instances meet, accumulators might be moved
  };
  for (;;) {
#pragma unroll
    for (int i = 0; i < kMT; ++i)
#pragma unroll
      for (int j = 0; j < kNT; ++j) acc[i][j] = f32x4{};
    // Group 1 runs one phase late.  From here on a barrier ends group 0's M phase and group 1's C
    // phase, the next one group 0's C phase and group 1's M phase, and so on.
    if (wm == 1) block_barrier();
    const long long clock0 = __builtin_amdgcn_s_memtime(), tick0 = __builtin_amdgcn_s_memrealtime();
    if (pairs == 4) k_loop(std::integral_constant<int, 8>{});
    else if (pairs == 3) k_loop(std::integral_constant<int, 6>{});
    else if (pairs == 2) k_loop(std::integral_constant<int, 4>{});
    else if (pairs == 1) k_loop(std::integral_constant<int, 2>{});
    else k_loop(std::integral_constant<int, 0>{});
    if (a.clocks != nullptr && t == 0 && tid == 0) {  // measurement aid: this wavefront's K loop
      a.clocks[0] = __builtin_amdgcn_s_memtime() - clock0;
      a.clocks[1] = __builtin_amdgcn_s_memrealtime() - tick0;
      a.clocks[2] = k_tiles;
    }
    if (left == 1) wait_loads_all();  // (of the requests of nothing: a workgroup does not end while a load into its LDS is under way)
    // The last M phase of both groups is over since group 0's last barrier, and the slot of the last activation rows, the next one to
    // be requested, holds the images: the two K-steps of the next tile that are under way or have landed lie in the others.
    if (a.bias != nullptr) epilogue(acc, first_row, mine, n0 + wn * kNT * 16, a_load, std::true_type{});
    else epilogue(acc, first_row, mine, n0 + wn * kNT * 16, a_load, std::false_type{});
    if (--left == 0) break;
    n0 += kBN;
    block_barrier();  // the images are read, their slot may be filled
  }
}

// The sum over experts of ceil(M_e / 256) never exceeds P / 256 + E; whole rounds of XCD patches.  What the loads leave of it is room for
// units, and of experts with a little over whole blocks each nothing is left, so there are as many workgroups as the end of a list of
// even loads needs (us, without them and with them: 60 x 274 rows 7608 -> 608 373 and 326, 16 x 296 rows 4032 -> 2312 139 and 120, 32 x 294
// rows 7448 -> 1096 344 and 276).  Room for the longest end of any list costs others more than it gives: 64 x 400 rows 768 -> 3072
// 141 -> 147 us, 16 x 2048 rows 4096 -> 1024 213 -> 218.
long workgroups_of_list(int P, int E, int tiles_n) {
  const long used = std::min(E, P), rows = used > 0 ? (P + used - 1) / used : 0, over = rows % kBM;
  const long even = (rows + kBM - 1) / kBM * used * tiles_n;
  GemmArgs any{};
  any.tiles_n = tiles_n;
  any.grid = 0x7fffffff;
  long entries = (static_cast<long>(P + kBM - 1) / kBM + E) * tiles_n;
  if (even <= kMostRounds * kRound)
    entries = std::max(entries, even + 3 * end_of_list(any, static_cast<int>(even), over > 0 && over <= kFewRows ? static_cast<int>(used) : 0,
                                                       [=](int n) { return n / tiles_n; }).cut);
  return (entries + kRound - 1) / kRound * kRound;
}

// A list of up to `entries` tiles of which whole rounds are walked, `walk` tiles to a workgroup: the workgroups it needs at most, with
// the units of an end that is cut and one to clear row tags.  (A list one tile short of another walked round needs more than a longer one.)
long workgroups_that_walk(long entries, int walk) {
  const long per = static_cast<long>(walk) * kRound, rounds = entries / per;
  const long most = rounds == 0 ? entries : std::max(entries - rounds * (per - kRound), rounds * kRound + per - kRound - 1);
  return std::min(entries, (most + 4 * kMostCutOfFewRows + 1 + kRound - 1) / kRound * kRound);
}

// Column tiles that a workgroup of the whole rounds walks: 2, or where their number is odd 3 or 5.  A walked tile costs neither a look
// at the loads nor a wait for its first K-steps nor the end of a workgroup, 4 us of the 33 that a tile of K = 1024 takes (us, one tile a workgroup
// and this many: 64 x 300 rows 768 -> 3072 + GELU 153 and 140, skewed top-2 rows of 32 experts 1024 -> 4096 + GELU 155 and 149, 16 x 2048 rows
// 256 -> 1024 34.0 and 31.2, 8 x 4000 rows 768 -> 768 46.3 and 45.3; 128 experts of ragged loads 1024 -> 4096 389 and 361).  With 4 of them even loads of
// many rounds gain another 1 to 2 % (512 -> 2048 85.7 and 84.5), skewed ones lose 3 to 6 (158 for the 149).  Where K is long there is
// little to win and there are few column tiles, of which then fewer row blocks of an XCD share the weights: 16 skewed experts of 32768 rows
// 4096 -> 1024 222 and 235, 1024 -> 1024 63.3 and 61.4, 4096 -> 2048 417 and 411, 8 x 4096 rows 8192 -> 2048 762 and 771.
int walk_of_list(const GemmArgs& a) {
  if (a.K % kBK != 0 || a.K > (a.tiles_n < 8 ? 1024 : 4096)) return 1;
  for (int w : {2, 3, 5})
    if (a.tiles_n % w == 0) return w;
  return 1;
}

// Fills in how the list of tiles is laid out and walked; the workgroups to launch.
long plan_list(GemmArgs& a) {
  a.tiles_n = (a.N + kBN - 1) / kBN;
  const long grid = workgroups_of_list(a.P, a.E, a.tiles_n);
  // The timed form wants the clocks of a whole tile, also of a list that would be cut to the last: it is told of no workgroups for units.
  // (A test of a.clocks in the kernel itself cost 32768 rows of 16 experts 1024 -> 4096 -> 1024 7 us of 577.)
  a.grid = a.clocks != nullptr ? 0 : static_cast<int>(grid);
  a.tiles_n_inverse = 0xffffffffu / static_cast<uint32_t>(a.tiles_n);
  a.walk = a.clocks != nullptr ? 1 : walk_of_list(a);
  a.walk_inverse = 0xffffffffu / static_cast<uint32_t>(a.walk);
  return a.walk > 1 ? workgroups_that_walk(grid, a.walk) : grid;
}

template <int ACT, bool ROUTED, bool OUTF32>
int launch_pingpong(GemmArgs& a, hipStream_t st) {
  const long grid = plan_list(a);
  auto* fn = &grouped_gemm_pingpong_kernel<ACT, ROUTED, OUTF32>;
  if (const int rc = allow_dynamic_lds(reinterpret_cast<const void*>(fn), kLdsBytes); rc != BRT_OK) return rc;
  hipLaunchKernelGGL(fn, dim3(static_cast<unsigned>(grid)), dim3(kWaves * 64), kLdsBytes, st, a);
  return check_launch("grouped_gemm_pingpong_kernel");
}

}  // namespace

// Shapes the ping-pong tiles take: K of at least two K-steps of 64, widths that keep the offsets inside a tile within 32 bits; every form but the
// weighted accumulate.
constexpr int kMostWidth = 1 << 20;
bool pingpong_gemm_applies(const GemmArgs& a) { return a.gates == nullptr && a.K >= 2 * kBK && a.K <= kMostWidth && a.N <= kMostWidth; }

template <int ACT>
int launch_pingpong_form(GemmArgs& a, hipStream_t st) {
  const bool f32 = a.out_f32 != nullptr;
  if (a.tags != nullptr) return f32 ? launch_pingpong<ACT, true, true>(a, st) : launch_pingpong<ACT, true, false>(a, st);
  return f32 ? launch_pingpong<ACT, false, true>(a, st) : launch_pingpong<ACT, false, false>(a, st);
}

int launch_pingpong_gemm(GemmArgs& a, int act, hipStream_t st) {
  // Rows that are no whole 64-byte pieces are written with ordinary stores whatever their size: the pieces of neighbouring
  // wavefronts that lie in one of them meet in the L2 (us, streamed and not: 16 x 500 rows 936 -> 1872 43.0 and 38.2, 16 x 2000 rows
  // 1000 -> 2000 163 and 149, 32 x 1000 rows 520 -> 1040 81 and 74, 16 x 2048 rows 1024 -> 4104 319 and 313; whole pieces, 4 x 8000
  // rows 1992 -> 7968, 941 and 1020; fp32 rows 16 x 1732 rows 640 -> 984 74 and 53, 32 x 298 rows 272 -> 2088 63 and 43, 32 x 1000 rows
  // 1024 -> 4104 367 and 320).  On the 160-row kernel it is level or loses (12 x 140 rows 1800 -> 7208 140 and 143).
  if (a.N % (a.out_f32 != nullptr ? 16 : 32) != 0) a.plain_out = 1;
  if (act == BRT_ACT_GELU) return launch_pingpong_form<BRT_ACT_GELU>(a, st);
  if (act == BRT_ACT_RELU) return launch_pingpong_form<BRT_ACT_RELU>(a, st);
  return launch_pingpong_form<BRT_ACT_NONE>(a, st);
}

}  // namespace brt

extern "C" int brt_hip_grouped_gemm_tiles_cut(const int32_t* loads, int E, int P, int N, int row_tags) {
  using namespace brt;
  if (!loads || E <= 0 || P < 0 || N <= 0) return fail(BRT_E_INVALID, "bad arguments E=%d P=%d N=%d", E, P, N);
  GemmArgs a{};
  int some_tag = 0;
  a.tiles_n = (N + kBN - 1) / kBN;
  a.grid = static_cast<int>(workgroups_of_list(P, E, a.tiles_n));
  a.row_tags_out = row_tags ? &some_tag : nullptr;
  long blocks = 0;
  int few = 0;
  for (int e = 0; e < E; ++e) {
    if (loads[e] < 0) return fail(BRT_E_INVALID, "expert %d has %d rows", e, loads[e]);
    const int over = loads[e] % kBM;
    blocks += (loads[e] + kBM - 1) / kBM;
    few += over > 0 && over <= kFewRows;
  }
  if (blocks * a.tiles_n > 0x7fffffffll) return fail(BRT_E_INVALID, "%ld row blocks of %d tiles", blocks, a.tiles_n);
  return end_of_list(a, static_cast<int>(blocks * a.tiles_n), few, [&](int n) { return n / a.tiles_n; }).cut;
}

extern "C" int brt_hip_grouped_gemm_walk(int E, int P, int K, int N, int* workgroups) {
  using namespace brt;
  if (!workgroups || E <= 0 || P <= 0 || K <= 0 || N <= 0) return fail(BRT_E_INVALID, "bad arguments E=%d P=%d K=%d N=%d", E, P, K, N);
  GemmArgs a{};
  a.E = E; a.P = P; a.K = K; a.N = N;
  *workgroups = static_cast<int>(plan_list(a));
  return a.walk;
}
