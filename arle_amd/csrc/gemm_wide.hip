// bfloat16 matrix product for prompt portions:  C[M,N] = X[M,K] . W[N,K]^T, both row-major, K a multiple of 64.
//
// A workgroup owns BM rows x BN columns (64 to 256 x 64 to 320) and walks K in stages of 64: the stage's rows of X and W, 128
// bytes each, go from memory straight into LDS (global_load_lds, no registers on the way), two to five stages deep, and every
// wave feeds v_mfma_f32_32x32x16_bf16 from there.  What bounds it, and what was done about that (MI355X, gate|up of the
// Qwen3-4B shape, N 19,456, K 2,560, weights cold):
//
//   * The matrix cores, at the clock that the chip holds when all 256 compute units multiply real data (1.75 to 1.84 PFLOP/s):
//     the loop alone runs at 1.53, a whole launch of 8,192 rows at 1.25 (652 us; the library's product and the activation
//     kernel 763, gemm_tiles 760; cards differ by 7 %).
//   * Turns: a launch lasts as many turns of its workgroups as they fill the compute units.  gate|up at 2,048 rows is 608
//     tiles of 256 x 256, three turns for 2.4; 256 x 320 is 488, two turns for 1.9: 172 us against gemm_tiles' 222.  So there are
//     nineteen shapes, and the caller's plan takes the one whose turns are shortest (ops.wide_plan).
//   * Few rows: W streams at what the workgroups have in flight.  Shapes whose stages are small keep three to five of them in the
//     LDS (80 to 150 KB): a stage's fetch has two to four stages' time.  9 to 256 rows are then W at 4 to 4.6 TB/s: 64 rows 26.3 us
//     with two stages and lines touched ahead 32.7 (128 x 96, 97 rows: 30.6 / 34.9; 128 x 160, 160 rows 33.4 / 37.7); a sixth stage and
//     more change nothing.  From operand tiles, whose kilobytes lie whole in memory where rows are 128 bytes each 5 KB apart,
//     64 rows take 23.7 us for 26.8, 128 rows 29.5 for 32.7, 256 rows 35.0 for 38.7; from 544 rows on the two are level.
//   * Weights that one row block reads (ONCE) are loaded past the caches, from tiles and from rows (a load takes whole lines of either).
//     Cold, us, kept / past: 24,576 x 4,096 with the activation, 33 rows, 40.1 / 36.6 from tiles and 47.2 / 42.7 from rows; 4,096 x 12,288 in
//     three parts 24.3 / 22.6 and 25.9 / 24.4; 128 rows level to 4 % ahead.  Whole steps of the Qwen3-4B shape, means of four to eight
//     engines of each (which differ by 2 % among themselves): prompts of 33 and 64 tokens 2,686 / 2,587 and 2,998 / 2,891, 64 requests
//     5,760 / 5,698; prompts of 97 and 120 tokens (3,357 / 3,319, 3,524 / 3,506) and 19 requests (2,906 / 2,895) within the spread.
//   * Latency of what comes from memory in the large shapes: with two stages a fetch has one stage's time (1.2 to 1.8 us), which
//     a miss of the L2 under load does not keep to.  There every wave touches, four stages ahead, a few of the 128-byte lines that its
//     XCD's workgroups will fetch (a dword a line, into a corner of LDS that nobody reads): 2,048 rows 223 -> 186 us, 8,192
//     rows 679 -> 600 in the form that the kernel had then.  More stages of 32 k instead (rows of 64 bytes) were 6 to 8 % slower: half lines cost the fetch path
//     twice the requests.
//   * The step's operand reads (4 cycles of LDS each) and loads are pinned between its products (sched_barrier): the next
//     step's operands are read while this step multiplies, the barrier of a stage stands in its last step, behind which
//     the first operands of the next stage are read and the place of this one is filled again.
//   * The activation of a workgroup's 40 thousand pairs: the same error as expf and a divide without their cases for what
//     leaves the floats, 167 us at 2,048 rows where the bare exponential and reciprocal of the vector unit (errors up to 63
//     ulp below zero) take 163 in the same run.
//
// Four waves (one a SIMD) or eight, measured alike in the loop; eight hold the accumulators of 256 x 320 in 256 registers each.
#include "common.h"

#include <type_traits>

namespace arle {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWdXcds = 8;
constexpr int kWdXcdPlaces = 32;   // workgroups that an XCD runs at a time: one a compute unit
constexpr int kWdPatchRows = 8, kWdPatchCols = 4;   // row and column blocks of a patch (see the kernel)
constexpr int kWdK = 64;           // k of a stage: rows of 128 bytes
constexpr int kEpiNone = 0, kEpiSiluMul = 1;

struct WideArgs {
  const uint16_t* x;
  int64_t ldx;
  const uint16_t* w;
  int64_t ldw;
  void* out;
  int64_t ldo;
  int M, N, K;
  int m_blocks, n_blocks;
  int stages_per_split;
  int64_t split_stride;
  int tiled;               // w holds operand tiles (see below) instead of rows
};

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // m0 is a reserved register: naming it as clobbered is the point
// 16 bytes a lane from base + lane_bytes to lds_at + 16 lane.  As assembly, because behind the builtin every LDS read is
// made to wait for all loads in flight.
__device__ __forceinline__ void wide_load(const uint16_t* base, uint32_t lane_bytes, uint32_t lds_at) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_at), "v"(lane_bytes), "s"(base)
               : "memory", "m0");
}
// The same for what no other workgroup reads: past the caches, where it would only displace what is read again.
__device__ __forceinline__ void wide_load_once(const uint16_t* base, uint32_t lane_bytes, uint32_t lds_at) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(lds_at), "v"(lane_bytes), "s"(base)
               : "memory", "m0");
}
// A dword of each lane's line, to a place in LDS that nobody reads: it brings the line into the L2.
__device__ __forceinline__ void wide_touch(const uint16_t* from, uint32_t lds_at) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(lds_at), "v"(from) : "memory", "m0");
}
#pragma clang diagnostic pop

// x / (1 + exp(-x)) to the error of expf and a whole divide, for |x| < kSiluNear, where nothing leaves the range of a
// float: exp(-x) = 2^t (1 + r), t = -x log2(e) rounded and r = -x - t ln 2, ln 2 in two parts; the quotient by 1 + 2^t from the
// reciprocal, corrected by what is left of x behind it and behind its share of 2^t r.  Against 64 bits over [-80, 80]: at most
// 2.71 ulp, 0.44 to 0.65 in the root mean square, for both forms alike (the vector unit's exponential of t alone and its
// reciprocal, as they come: up to 63 ulp, 21).
constexpr float kSiluNear = 80.0f;
__device__ __forceinline__ float silu_near(float x) {
#pragma clang fp contract(off)
  constexpr float kLog2e = 1.44269502162933349609375f, kLn2Hi = 0.693147182464599609375f, kLn2Lo = -1.904654212125933550e-9f;
  const float t = x * -kLog2e, r = fmaf(t, -kLn2Lo, fmaf(t, -kLn2Hi, -x));
  const float e = __builtin_amdgcn_exp2f(t), d = 1.0f + e;
  const float inv = __builtin_amdgcn_rcpf(d), q = x * inv;
  return fmaf(fmaf(-(e * r), q, fmaf(-d, q, x)), inv, q);
}
__device__ __forceinline__ float silu_whole(float x) { return x / (1.0f + expf(-x)); }

template <int WM, int WN, int TM, int TN, int NS, int EPI, typename TOut, bool ONCE>
__global__ __launch_bounds__(WM* WN* kWave, (WM * WN + 3) / 4) void gemm_wide_kernel(const WideArgs a) {
  constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN, kWaves = WM * WN;
  constexpr int kRowsALoad = 8 * kWaves;                        // rows that one load of every wave brings
  static_assert(BM % kRowsALoad == 0 && BN % kRowsALoad == 0 && kRowsALoad % 16 == 0, "whole loads, of whole rounds of the pieces' order");
  constexpr int LX = BM / kRowsALoad, LA = (BM + BN) / kRowsALoad;
  constexpr int kStage = (BM + BN) * 128;
  constexpr int kProducts = TM * TN, kReads = TM + TN;
  constexpr int kSlots = kProducts > 1 ? kProducts - 1 : 1, kReadsASlot = (kReads + kSlots - 1) / kSlots;   // reads go behind the products 1, 2, ... (behind the only one)
  constexpr bool kTouch = NS == 2;
  static_assert(!ONCE || !kTouch, "lines that are touched ahead have to stay in the L2");
  extern __shared__ __align__(16) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, h = lane >> 5;
  const int wm = wave / WN, wn = wave % WN;

  // Column blocks go to the XCDs in turn.  An XCD takes its own in groups of kWdPatchCols, a group's row blocks in patches of
  // kWdPatchRows, and a patch column by column; patches at the ends are as small as they have to be and leave no place empty:
  // workgroups go to an XCD's four shader engines in turn, those that leave at once too, and with ten row blocks as 8 + 2
  // and six empty places two of the engines had nine workgroups for their eight units (4,096 columns, K 2,048, 1,280
  // rows: 49 us, against 29 without the empty places).
  const int xcd = blockIdx.x % kWdXcds, q = blockIdx.x / kWdXcds;
  const int col_group = q / (a.m_blocks * kWdPatchCols), in_group = q - col_group * a.m_blocks * kWdPatchCols;
  const int cols_here = min(kWdPatchCols, (a.n_blocks + kWdXcds - 1) / kWdXcds - col_group * kWdPatchCols);
  const int row_group = in_group / (kWdPatchRows * cols_here), in_patch = in_group - row_group * kWdPatchRows * cols_here;
  const int rows_here = min(kWdPatchRows, a.m_blocks - row_group * kWdPatchRows);
  const int patch_col = in_patch / rows_here, patch_row = __builtin_amdgcn_readfirstlane(in_patch - patch_col * rows_here);
  const int mb = __builtin_amdgcn_readfirstlane(row_group * kWdPatchRows + patch_row);
  const int nb = __builtin_amdgcn_readfirstlane((col_group * kWdPatchCols + patch_col) * kWdXcds + xcd);
  if (nb >= a.n_blocks) return;  // the whole workgroup
  const int m0 = mb * BM, n0 = nb * BN;
  const int M = a.M, N = a.N;
  const int all_stages = a.K / kWdK;
  const int st0 = blockIdx.y * a.stages_per_split;
  const int n_st = min(a.stages_per_split, all_stages - st0);
  const uint16_t* xb = a.x + static_cast<int64_t>(m0) * a.ldx + static_cast<int64_t>(st0) * kWdK;
  // a tile of W: 16 columns x 32 k, 1 KB; a stage's k of 16 columns are two of them side by side
  const int tile_row = a.K / 32 * 512;     // elements between the tiles of neighbouring sixteens of columns
  const int w_step = a.tiled ? 1024 : kWdK;
  const uint16_t* wb = a.tiled ? a.w + static_cast<int64_t>(n0 / 16) * tile_row + static_cast<int64_t>(st0) * w_step
                               : a.w + static_cast<int64_t>(n0) * a.ldw + static_cast<int64_t>(st0) * kWdK;

  // a load brings 8 rows of 128 bytes; piece lane % 8 of an LDS row holds the row's k piece (lane % 8) ^ (row / 2 % 8),
  // so that sixteen lanes of an operand read never share a bank
  const int lr = 8 * wave + (lane >> 3);
  const int piece = (lane & 7) ^ ((lr >> 1) & 7);
  uint32_t off[LA];
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const bool of_x = i < LX;
    const int row = kRowsALoad * (of_x ? i : i - LX) + lr;
    off[i] = static_cast<uint32_t>(min(row, of_x ? M - 1 - m0 : N - 1 - n0)) * static_cast<uint32_t>((of_x ? a.ldx : a.ldw) * 2) + piece * 16;
    if (!of_x && a.tiled) {      // a wave's load is a tile
      const int tile = (i - LX) * kWaves + wave;
      off[i] = static_cast<uint32_t>(min(tile / 2, (N - n0) / 16 - 1)) * static_cast<uint32_t>(tile_row * 2) + (tile % 2) * 1024 + lane * 16;
    }
  }
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)lds)) + 1024u * wave);
  auto load = [&](int i, uint32_t buf, const uint16_t* xs, const uint16_t* ws) {   // i is a constant where this is called
    if (i < LX || !ONCE) wide_load(i < LX ? xs : ws, off[i], lds0 + buf + 1024u * kWaves * i);
    else wide_load_once(ws, off[i], lds0 + buf + 1024u * kWaves * i);
  };
  // What comes from memory and not from the L2 comes late: every stage a wave touches a few of the 128-byte lines that the
  // stage kAhead later will fetch (the workgroups that share a column block's weights or a row block's x in a patch
  // share out its lines), so that the fetch itself meets the L2.  A lane touches one line a stage, so a wave 64 of them: where a
  // patch has a single row block, the four waves of 256 and 320 columns have 64 and 80 lines of W each and no lane for x
  // (which the column blocks' workgroups of the XCD then fetch from the L2 behind whichever of them comes first).
  constexpr int kAhead = 4;      // with two stages only: three and more bring what comes late themselves
  const int x_share = a.m_blocks > kWdPatchRows ? kWdPatchCols : kWdXcdPlaces / rows_here;
  const int w_lines = (BN + rows_here * kWaves - 1) / (rows_here * kWaves), x_lines = (BM + x_share * kWaves - 1) / (x_share * kWaves);
  const uint16_t* touch_from;
  int touch_step = kWdK;
  if (lane < w_lines) {
    const int line = min((patch_row * kWaves + wave) * w_lines + lane, N - 1 - n0);
    touch_from = wb + (a.tiled ? static_cast<int64_t>(line / 16) * tile_row + line % 16 * 64 : static_cast<int64_t>(line) * a.ldw);
    touch_step = w_step;
  } else {
    touch_from = xb + static_cast<int64_t>(min((((nb / kWdXcds) % x_share) * kWaves + wave) * x_lines + min(lane - w_lines, x_lines - 1), M - 1 - m0)) * a.ldx;
  }
  const bool touches = lane < w_lines + x_lines;
  const uint32_t touch_at = __builtin_amdgcn_readfirstlane(
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)lds)) + NS * kStage + 256u * wave);
  auto touch = [&](int stages) {
    if (touches) wide_touch(touch_from + stages * touch_step, touch_at);
  };
  uint32_t at[4], w_piece[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    at[kk] = j * 128 + (((2 * kk + h) ^ ((j >> 1) & 7)) * 16);
    w_piece[kk] = a.tiled ? (j >> 4) * 2048 + kk * 512 + h * 256 + (j & 15) * 16 : at[kk];   // 16 lanes read 256 bytes side by side
  }
  const uint32_t x_at = wm * TM * 4096, w_at = BM * 128 + wn * TN * 4096;

  f32x16 acc[TM][TN];
#pragma unroll
  for (int t = 0; t < TM; ++t)
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t][tn][r] = 0.f;
  bf16x8 fx[2][TM], fw[2][TN];
  auto read_one = [&](int i, int set, int kk, uint32_t buf) {
    if (i < TM)
      fx[set][i] = *reinterpret_cast<const bf16x8*>(lds + buf + x_at + at[kk] + 4096 * i);
    else
      fw[set][i - TM] = *reinterpret_cast<const bf16x8*>(lds + buf + w_at + w_piece[kk] + 4096 * (i - TM));
  };

  constexpr int kEarly = (LA + 1) / 2;   // loads of a stage that go out in the step that frees its place; the others in the step after it
  static_assert((NS - 2) * LA + kEarly < 64, "the loads in flight fit the counter");
#pragma unroll
  for (int st = 0; st < NS - 1; ++st) {
    if (st < n_st) {
#pragma unroll
      for (int i = 0; i < LA; ++i) load(i, st * kStage, xb + st * kWdK, wb + st * w_step);
    }
  }
  if (n_st >= NS) {
#pragma unroll
    for (int i = 0; i < kEarly; ++i) load(i, (NS - 1) * kStage, xb + (NS - 1) * kWdK, wb + (NS - 1) * w_step);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * LA + kEarly) : "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  if (kTouch && n_st > 3) touch(2), touch(3);
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < kReads; ++i) read_one(i, 0, 0, 0);

  // One stage, four steps of 16 k, and what it sends for later: the rest of stage s + NS - 1 in its first step, to the place
  // of the stage before it, and the first part of s + NS in its last, to its own.  LEFT: the stages that follow it, up to NS.
  // TOUCH: it touches the lines of stage s + kAhead.
  uint32_t before = (NS - 1) * kStage, buf = 0, next = kStage;
  auto stage = [&](auto left_tag, auto touch_tag) {
    constexpr int LEFT = decltype(left_tag)::value;
    constexpr bool TOUCH = decltype(touch_tag)::value;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int set = kk & 1;
#pragma unroll
      for (int m = 0; m < kProducts; ++m) {
        if (kk == 3 && m == (kProducts > 1 ? 1 : 0) && LEFT > 0) {
          // every wave has its operands of this stage, and its pieces of the next one have landed: what was sent behind those
          // may still be on its way
          constexpr int kFlying = (LEFT - 1 < NS - 2 ? LEFT - 1 : NS - 2) * LA + (TOUCH ? 1 : 0);
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LEFT > 0 ? kFlying : 0) : "memory");
          __builtin_amdgcn_s_barrier();
          __builtin_amdgcn_sched_barrier(0);
        }
        const int t = m % TM, tn = m / TM;
        acc[t][tn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw[set][tn], fx[set][t], acc[t][tn], 0, 0, 0);
        // the next step's operands
        const int slot = kProducts > 1 ? m - 1 : 0;
#pragma unroll
        for (int r = slot * kReadsASlot; slot >= 0 && r < (slot + 1) * kReadsASlot && r < kReads; ++r) {
          if (kk < 3) read_one(r, set ^ 1, kk + 1, buf);
          else if (LEFT > 0) read_one(r, set ^ 1, 0, next);
        }
        if (kk == 3 && LEFT >= NS && slot >= 0) {
#pragma unroll
          for (int i = 0; i < kEarly; ++i)
            if (i * kSlots / kEarly == slot) load(i, buf, xb + NS * kWdK, wb + NS * w_step);
        }
        if (kk == 0 && LEFT >= NS - 1) {
#pragma unroll
          for (int i = kEarly; i < LA; ++i)
            if ((i - kEarly) * kProducts / (LA - kEarly) == m) load(i, before, xb + (NS - 1) * kWdK, wb + (NS - 1) * w_step);
        }
        if (kk == 1 && TOUCH && slot == 0) touch(kAhead);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    before = buf, buf = next, next = next + kStage == NS * kStage ? 0 : next + kStage;
    xb += kWdK, wb += w_step;
  };
  constexpr std::false_type plain{};
  int s = 0;
  if constexpr (kTouch) {
    for (; s + kAhead < n_st; ++s) {
      stage(std::integral_constant<int, NS>{}, std::true_type{});
      touch_from += touch_step;
    }
  }
  for (; s + NS < n_st; ++s) stage(std::integral_constant<int, NS>{}, plain);
  const int left = n_st - 1 - s;
  static_assert(NS <= 5, "the last stages are written out");
  if constexpr (NS > 4) { if (left >= 4) stage(std::integral_constant<int, 4>{}, plain); }
  if constexpr (NS > 3) { if (left >= 3) stage(std::integral_constant<int, 3>{}, plain); }
  if constexpr (NS > 2) { if (left >= 2) stage(std::integral_constant<int, 2>{}, plain); }
  if (left >= 1) stage(std::integral_constant<int, 1>{}, plain);
  stage(std::integral_constant<int, 0>{}, plain);

  // acc[t][tn][r] = C[m0 + 32 (TM wm + t) + j][n0 + 32 (TN wn + tn) + 8 (r / 4) + 4 h + r % 4]; row tiles go through a
  // part of LDS of the wave's own (float32 ones a column tile at a time) and leave as whole rows
  constexpr int kElt = static_cast<int>(sizeof(TOut));
  constexpr int kTile = EPI == kEpiSiluMul ? 16 : 32;                // output columns of a column tile
  constexpr int kGroup = kElt == 2 ? TN : 1;                         // column tiles that leave together
  constexpr int kPitch = kTile * kGroup * kElt + 16;
  constexpr int kPieces = kTile * kGroup * kElt / 16;
  static_assert(kWaves * 32 * kPitch <= NS * kStage, "the epilogue's rows fit the stages");
  TOut* out = static_cast<TOut*>(a.out) + static_cast<int64_t>(blockIdx.y) * a.split_stride;
  const int n_out = EPI == kEpiSiluMul ? N / 2 : N;
  const int c0 = (EPI == kEpiSiluMul ? n0 / 2 : n0) + kTile * TN * wn;
  const int r0 = m0 + 32 * TM * wm;
  __syncthreads();
  unsigned char* mine = lds + wave * (32 * kPitch);
  // FAR: a gate of the wave is beyond kSiluNear.  That copy stands behind the other one: inside it, tile by tile, it took the
  // kernel from 20 to 47 KB, and between a model's other kernels a launch waits for its code.
  auto leave = [&](auto far_tag) {
    constexpr bool FAR = decltype(far_tag)::value;
#pragma unroll
    for (int t = 0; t < TM; ++t) {
#pragma unroll
      for (int g = 0; g < TN; g += kGroup) {
#pragma unroll
        for (int tn = g; tn < g + kGroup; ++tn) {
#pragma unroll
          for (int q4 = 0; q4 < kTile / 8; ++q4) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              v[e] = acc[t][tn][4 * q4 + e];
              if constexpr (EPI == kEpiSiluMul) v[e] = (FAR ? silu_whole(v[e]) : silu_near(v[e])) * acc[t][tn][4 * q4 + e + 8];
            }
            unsigned char* to = mine + j * kPitch + (kTile * (tn - g) + 8 * q4 + 4 * h) * kElt;
            if constexpr (kElt == 2)
              *reinterpret_cast<uint2*>(to) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
            else
              *reinterpret_cast<float4*>(to) = float4{v[0], v[1], v[2], v[3]};
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int i = 0; i < kPieces / 2; ++i) {
          const int idx = 64 * i + lane, rr = idx / kPieces, pc = idx % kPieces;
          const u32x4 v = *reinterpret_cast<const u32x4*>(mine + rr * kPitch + pc * 16);
          const int row = r0 + 32 * t + rr, col = c0 + kTile * g + pc * (16 / kElt);
          if (row < M && col < n_out) *reinterpret_cast<u32x4*>(out + static_cast<int64_t>(row) * a.ldo + col) = v;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
    }
  };
  float most = 0.f;
  if constexpr (EPI == kEpiSiluMul) {
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int e = 0; e < 8; ++e) most = fmaxf(most, fabsf(acc[t][tn][e]));   // a NaN may pass: it stays one either way
  }
  if (__builtin_expect(EPI != kEpiSiluMul || !__any(most >= kSiluNear), 1)) leave(std::false_type{});
  else if constexpr (EPI == kEpiSiluMul) leave(std::true_type{});
}

template <int WM, int WN, int TM, int TN, int NS, int EPI, typename TOut, bool ONCE>
int launch_wide_as(WideArgs a, int splits, hipStream_t s) {
  constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN;
  constexpr size_t lds = NS * (BM + BN) * 128 + (NS == 2 ? 256 * WM * WN : 0);
  static_assert(lds <= 160 * 1024, "the stages fit the LDS");
  static OnceADevice asked;
  if (const int e = ask_lds(asked, lds, {reinterpret_cast<const void*>(&gemm_wide_kernel<WM, WN, TM, TN, NS, EPI, TOut, ONCE>)})) return e;
  a.m_blocks = (a.M + BM - 1) / BM;
  a.n_blocks = (a.N + BN - 1) / BN;
  const long long grid = static_cast<long long>(a.m_blocks) * ((a.n_blocks + kWdXcds - 1) / kWdXcds) * kWdXcds;
  if (grid > 0x7fffffffLL) return static_cast<int>(hipErrorInvalidValue);
  gemm_wide_kernel<WM, WN, TM, TN, NS, EPI, TOut, ONCE><<<dim3(static_cast<unsigned>(grid), static_cast<unsigned>(splits)), WM * WN * kWave, lds, s>>>(a);
  return launch_status();
}

// ONCE where there is one row block: with several, the workgroups of a column block meet in their XCD's L2.
template <int WM, int WN, int TM, int TN, int NS, int EPI, typename TOut>
int launch_wide(const WideArgs& a, int splits, hipStream_t s) {
  if constexpr (NS > 2) {
    if (a.M <= 32 * WM * TM) return launch_wide_as<WM, WN, TM, TN, NS, EPI, TOut, true>(a, splits, s);
  }
  return launch_wide_as<WM, WN, TM, TN, NS, EPI, TOut, false>(a, splits, s);
}

template <int WM, int WN, int TM, int TN, int NS>
int dispatch_wide(const WideArgs& a, int splits, int out_dtype, int epilogue, hipStream_t s) {
  if (epilogue) return launch_wide<WM, WN, TM, TN, NS, kEpiSiluMul, bf16>(a, splits, s);
  return out_dtype == kF32 ? launch_wide<WM, WN, TM, TN, NS, kEpiNone, float>(a, splits, s) : launch_wide<WM, WN, TM, TN, NS, kEpiNone, bf16>(a, splits, s);
}

}  // namespace arle

using namespace arle;

// x [M, K], w [N, K] bfloat16 with 16-byte aligned rows, K % 64 == 0, N % 32 == 0.  out [M, N] (bfloat16 or float32), or
// with epilogue 1 [M, N/2] bfloat16 (gate and up rows of w interleaved in blocks of 16): silu(gate) * up.  tiled: w is the
// operand tiles of [N, K], [N/16][K/32][64 lanes][8], lane 16 g + i = W[16 t + i][32 s + 8 g .. +7] (ldw is not looked at).
extern "C" int arle_gemm_wide(const void* x, long long ldx, const void* w, long long ldw, void* out, long long ldo, int out_dtype,
                              int M, int N, int K, int epilogue, int row_tiles, int col_tiles, int splits, int stages_per_split,
                              long long split_stride, int tiled, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  const int per16 = out_dtype == kF32 ? 4 : 8;
  if (K <= 0 || K % kWdK != 0 || N % 32 != 0 || ldx % 8 != 0 || ldw % 8 != 0 || ldx >= (1 << 20) || ldw >= (1 << 20) ||
      !aligned(x) || !aligned(w) || !aligned(out) || ldo % per16 != 0 || split_stride % per16 != 0 ||
      (epilogue != kEpiNone && epilogue != kEpiSiluMul) || (epilogue == kEpiSiluMul && out_dtype == kF32) || splits < 1 ||
      splits > 65535 || stages_per_split < 1 || (splits > 1 && (out_dtype != kF32 || epilogue != kEpiNone)))
    return static_cast<int>(hipErrorInvalidValue);
  const int stages = K / kWdK;
  if (static_cast<long long>(splits - 1) * stages_per_split >= stages || static_cast<long long>(splits) * stages_per_split < stages)
    return static_cast<int>(hipErrorInvalidValue);
  const WideArgs a{static_cast<const uint16_t*>(x), ldx, static_cast<const uint16_t*>(w), ldw, out, ldo, M, N, K,
                   0, 0, stages_per_split, split_stride, tiled};
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (1000 * row_tiles + col_tiles) {   // rows and columns of a workgroup
    case 64064: return dispatch_wide<2, 2, 1, 1, 5>(a, splits, out_dtype, epilogue, s);
    case 64096: return dispatch_wide<2, 1, 1, 3, 4>(a, splits, out_dtype, epilogue, s);
    case 64128: return dispatch_wide<2, 2, 1, 2, 4>(a, splits, out_dtype, epilogue, s);
    case 128064: return dispatch_wide<2, 2, 2, 1, 4>(a, splits, out_dtype, epilogue, s);
    case 128096: return dispatch_wide<4, 1, 1, 3, 4>(a, splits, out_dtype, epilogue, s);
    case 128128: return dispatch_wide<2, 2, 2, 2, 4>(a, splits, out_dtype, epilogue, s);
    case 128160: return dispatch_wide<4, 1, 1, 5, 3>(a, splits, out_dtype, epilogue, s);
    case 128192: return dispatch_wide<2, 2, 2, 3, 3>(a, splits, out_dtype, epilogue, s);
    case 128256: return dispatch_wide<2, 2, 2, 4, 3>(a, splits, out_dtype, epilogue, s);
    case 128320: return dispatch_wide<2, 2, 2, 5, 2>(a, splits, out_dtype, epilogue, s);
    case 192128: return dispatch_wide<2, 2, 3, 2, 3>(a, splits, out_dtype, epilogue, s);
    case 192192: return dispatch_wide<2, 2, 3, 3, 3>(a, splits, out_dtype, epilogue, s);
    case 192256: return dispatch_wide<2, 2, 3, 4, 2>(a, splits, out_dtype, epilogue, s);
    case 192320: return dispatch_wide<2, 2, 3, 5, 2>(a, splits, out_dtype, epilogue, s);
    case 256128: return dispatch_wide<4, 2, 2, 2, 3>(a, splits, out_dtype, epilogue, s);
    case 256160: return dispatch_wide<4, 1, 2, 5, 3>(a, splits, out_dtype, epilogue, s);
    case 256192: return dispatch_wide<4, 2, 2, 3, 2>(a, splits, out_dtype, epilogue, s);
    case 256256: return dispatch_wide<4, 2, 2, 4, 2>(a, splits, out_dtype, epilogue, s);
    case 256320: return dispatch_wide<4, 2, 2, 5, 2>(a, splits, out_dtype, epilogue, s);
  }
  return static_cast<int>(hipErrorInvalidValue);
}
