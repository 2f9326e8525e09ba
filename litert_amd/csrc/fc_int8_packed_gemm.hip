// Prefill-regime FULLY_CONNECTED on the re-tiled int8 filter: a dense int8 GEMM on the
// gfx950 matrix cores (v_mfma_i32_32x32x32_i8, the int8 instruction with the highest rate)
// that shares its weight layout with the decode GEMV, so a filter is kept in ONE form for
// every batch size.
//
//   out[m, n] = epilogue(sum_k x[m, k] * w[n, k])        x [M, K] row-major int8
//
// The filter is stored in 1 KiB tiles of 16 channels x 64 depth (lane L of a tile: channel
// L % 16, depth 16 * (L / 16) .. +16). A 32x32x32 operand (lane L: channel L % 32, 16 depth
// bytes of half L / 32) is gathered from two such tiles by per-lane addresses; each quarter
// of the wavefront still reads 256 consecutive bytes, so the load is as efficient as a
// contiguous one. Each wavefront owns 64 output channels and loads their operands straight
// from global memory into registers, two depth steps ahead -- the weights never touch LDS,
// because no other wavefront of the workgroup needs them. Only the activation rows are
// shared: the workgroup stages 128 rows x 128 depth per step in LDS (two buffers, rows padded
// to 144 bytes so that the 16-byte operand reads are conflict-free; 128 bytes of a row are one
// whole cache line) and every wavefront reads its sixteen operands from there. Per step and
// wavefront: 12 global loads, 16 LDS reads, 4 LDS writes, 32 MFMAs (1024 matrix-core cycles)
// and one barrier, all dealt out singly between the MFMAs: a wavefront is alone on its SIMD,
// so whatever holds up its instruction stream idles the matrix pipe.
// Launches that this 128 x 256 tile would cut into fewer workgroups than half the chip's CUs
// (batches of a few dozen to a few hundred rows), and short walks, run the same kernel with 64 or 128
// rows x 128 channels per workgroup (32 channels per wavefront).
//
// The outputs of a tile are put together in LDS (the row buffers, free by then) and stored in
// 16-byte pieces, whole cache lines per row.
//
// int32 accumulation is exact, so tiling cannot change the accumulator; bit-exactness rests
// on the epilogues, which are the ones of the GEMV kernels (fc_epilogues.h).
#include <type_traits>
#include <utility>

#include "fc_epilogues.h"
#include "kernels.h"

namespace lrtfc {
namespace {

using i32x16 = int __attribute__((ext_vector_type(16)));

constexpr int kThreads = 256;
constexpr int kWaves = 4;
constexpr int kSlab = 64;                     // depth of one tile of the packed filter
constexpr int kStep = 128;                    // depth per step: two slabs, one cache line of a row
constexpr int kXStride = kStep + 16;          // padded LDS row
constexpr int kSub = kStep / 32;              // MFMA depth sub-steps per step
constexpr int kGroupM = 4;                    // M-tiles per rasterization group

// f(std::integral_constant<int, 0>{}), f(<1>), ... : a loop whose index is a constant in
// every iteration, so that register arrays indexed by it stay in fixed registers.
template <int... Is, typename F>
__device__ __forceinline__ void ForEachConst(std::integer_sequence<int, Is...>, F&& f) {
  (f(std::integral_constant<int, Is>{}), ...);
}

// BM: batch rows per workgroup (128, or 64 for launches the large tile would leave with few
// workgroups); kWaveTiles: 32-channel MFMA tiles per wavefront (2 or 1); kRagged: the depth is no
// multiple of 16, so the last piece of every row is shifted into place on its way to LDS (a
// form of its own: a test for it inside the steps would break their straight line).
// kSlots: steps ahead at which weights are requested, one register set each (rows: one step less ahead
// of their way to LDS).
template <Int8Epilogue EPI, int BM, int kWaveTiles, bool kRagged, int kSlots>
__global__ __launch_bounds__(kThreads, 1) void FcInt8PackedGemmKernel(FcInt8Args a) {
  constexpr int BN = kWaves * kWaveTiles * 32;  // output channels per workgroup
  constexpr int kStageBytes = BM * kXStride;
  constexpr int kBatchTiles = BM / 32;
  constexpr int kXChunks = BM / 32;  // 16-byte chunks of activations a thread stages per step
  static_assert(BM % 64 == 0 && BN <= kThreads, "tile shape");
  __shared__ __align__(16) int8_t smem[2 * kStageBytes];
  __shared__ i32x4 chan_params[BN];  // per output channel of the tile, for the epilogue
  const int M = a.batches, N = a.out_depth, K = a.depth;
  const int slabs = (K + kSlab - 1) / kSlab;
  const int steps = (slabs + 1) / 2;
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  const int total = tiles_m * tiles_n;
  // The arguments that the first loads need, in registers ahead of the tile's arithmetic: the compiler reads
  // them behind it otherwise, and the workgroup waits once more (2048 x 4096 -> 4096 33.8 us, so 33.5).
  if (EPI == Int8Epilogue::kRequantize) {
    asm volatile("" ::"s"(a.multipliers), "s"(a.shifts), "s"(a.bias_i32), "s"(a.filter_row_sums),
                 "s"(a.per_channel), "s"(a.input_offset), "s"(a.output_offset), "s"(a.act_min),
                 "s"(a.act_max));
  } else {
    asm volatile("" ::"s"(a.per_channel_scales), "s"(a.bias_f32), "s"(a.zero_points), "s"(a.filter_row_sums));
  }
  asm volatile("" ::"s"(a.input), "s"(a.filter));

  // Workgroups are dealt round-robin to the 8 XCDs; give each XCD a contiguous range of tile
  // ids, ordered so that a range is a compact rectangle whose operands stay in that XCD's L2. The first
  // total % 8 XCDs have a tile more than the others. (Grids that are no multiple of 8 went unsorted: 5000
  // launches of 65 to 3000 rows, of which two thirds are such grids, us unsorted -> sorted: 64 x 128 tiles
  // 0.92 of the time in the mean, 128 x 128 0.95, 128 x 256 0.97; 1485 x 768 -> 9536, where 900 of the second
  // had taken the place of 456 of the third, 29.3 -> 23.8, with those 24.7.)
  const int xcd = static_cast<int>(blockIdx.x % 8);
  const int id = xcd * (total / 8) + min(xcd, total % 8) + static_cast<int>(blockIdx.x / 8);
  const int width = kGroupM * tiles_n;
  const int group = id / width;
  const int first_m = group * kGroupM;
  const int gsize = min(tiles_m - first_m, kGroupM);
  const int tm = first_m + (id % width) % gsize;
  const int tn = (id % width) / gsize;
  const int m0 = tm * BM, n0 = tn * BN;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // Per-channel epilogue inputs, one channel per thread, fetched now so that their latency
  // hides behind the main loop: {multiplier, shift, bias + input_offset * row_sum, rounding
  // term of the right shift} or {channel scale, bias, row sum, -}.
  i32x4 chan_p;
  bool plain_channel = true;  // this thread's channel allows the short requantization
  {
    const int n = min(n0 + tid, N - 1);
    i32x4 p = {0, 0, 0, 0};
    if (EPI == Int8Epilogue::kRequantize) {
      p[0] = a.per_channel ? a.multipliers[n] : a.multipliers[0];
      p[1] = a.per_channel ? a.shifts[n] : a.shifts[0];
      p[2] = a.bias_i32 ? a.bias_i32[n] : 0;
      if (a.input_offset != 0) p[2] += a.input_offset * a.filter_row_sums[n];
      p[3] = (p[1] < 0 && p[1] >= -31) ? (1 << (-p[1] - 1)) : 0;
      plain_channel = p[1] <= -1 && p[1] >= -31 && p[0] != INT32_MIN &&
                      p[2] > -(1 << 29) && p[2] < (1 << 29);
    } else {
      p[0] = __float_as_int(a.per_channel_scales ? a.per_channel_scales[n] : a.filter_scale);
      p[1] = __float_as_int(a.bias_f32 ? a.bias_f32[n] : 0.0f);
      p[2] = (EPI == Int8Epilogue::kHybrid && a.zero_points) ? a.filter_row_sums[n] : 0;
    }
    chan_p = p;
  }
  // EvalHybridDense's early exit for a whole-zero input (fully_connected.cc:789-795) matters only
  // where a bias element is -0.0f: a workgroup that stages such a channel settles the question
  // here, once, outside the loops that must unroll.
  bool zero_input = false;
  if (EPI == Int8Epilogue::kHybrid && a.zero_input_exit) {
    const bool mine = tid < BN && n0 + tid < N && a.bias_f32 != nullptr &&
                      IsNegativeZero(__int_as_float(chan_p[1]));
    if (__syncthreads_or(mine)) {
      zero_input = a.whole_input
                       ? WorkgroupAllZeroInt8(a.whole_input, static_cast<size_t>(a.whole_batches) * K)
                       : WorkgroupAllZeroInt8(a.input, static_cast<size_t>(M) * K);
    }
  }

  // Scale and zero point of the rows whose outputs this lane holds (row L % 32 of every batch tile).
  float row_scale[kBatchTiles];
  int32_t row_zero[kBatchTiles];
  bool small_zero = true;  // |zero point| < 2^23
#pragma unroll
  for (int j = 0; j < kBatchTiles; ++j) {
    row_scale[j] = 0.0f;
    row_zero[j] = 0;
    if (EPI != Int8Epilogue::kRequantize) {
      const int m = min(m0 + j * 32 + (lane & 31), M - 1);
      row_scale[j] = a.scaling_factors[m];
      if (a.zero_points) row_zero[j] = a.zero_points[m];
      small_zero = small_zero && row_zero[j] < (1 << 23) && row_zero[j] >= -(1 << 23);
    }
  }

  // Weight operands of this wavefront: lane L addresses channel L % 32 of MFMA tile i (tile
  // index clamped at the last 16-channel tile: duplicates are computed and never stored) and
  // the 16 bytes of depth half L / 32 within a 32-deep sub-step.
  const int ctiles = (N + 15) / 16;
  const int8_t* wp[kWaveTiles];
#pragma unroll
  for (int i = 0; i < kWaveTiles; ++i) {
    const int ct = min(n0 / 16 + (wave * kWaveTiles + i) * 2 + ((lane & 31) >> 4), ctiles - 1);
    wp[i] = a.filter + static_cast<size_t>(ct) * slabs * 1024 + (lane & 15) * 16 + (lane >> 5) * 256;
  }
  // Activation staging: 16-byte chunks per thread and step, chunk tid % 8 of rows tid / 8 + 32 p
  // (eight consecutive lanes read one whole 128-byte line of a row).
  const int ld_chunk = tid & 7;
  const int8_t* xp[kXChunks];
#pragma unroll
  for (int p = 0; p < kXChunks; ++p) {
    const int row = min(m0 + (tid >> 3) + 32 * p, M - 1);
    xp[p] = a.input + static_cast<size_t>(row) * K;
  }
  const int st_off = (tid >> 3) * kXStride + ld_chunk * 16;
  // An odd number of slabs leaves the second half of the last step without a filter tile: the
  // weight addresses are clamped to the last tile and the rows' half is staged as zeros.
  const bool upper_chunk = ld_chunk >= 4;
  // The piece a row ends in lies in this step and is shifted by this many bytes (kRagged).
  const int ragged_step = K / kStep;
  const int ragged_skip = RowPieceSkip(ragged_step * kStep + ld_chunk * 16, K);
  const int half_step = (slabs & 1) ? steps - 1 : -1;

  // Weights: wring[step % kSlots] holds a step's operands; a piece is requested again, for kSlots
  // steps later, right after the last MFMA that reads it. Rows: xr[step % kSlots], requested
  // kSlots + 1 steps before their use, staged two steps before it, read into fa during the step
  // before it.
  i32x4 wring[kSlots][kWaveTiles][kSub];
  i32x4 xr[kSlots][kXChunks];
  auto load_w_piece = [&](int step, auto slot, auto tile, auto sub) {
    constexpr int i = decltype(tile)::value, h = decltype(sub)::value;
    const int slab = min(2 * step + h / 2, slabs - 1);
    wring[decltype(slot)::value][i][h] = *reinterpret_cast<const i32x4*>(
        wp[i] + static_cast<size_t>(slab) * 1024 + (h & 1) * 512);
  };
  auto load_x_piece = [&](int step, auto set, auto piece) {
    // Past the end of a row (last partial slab, steps beyond the last) the address is clamped
    // into the row: whatever it reads meets zero padding in the packed filter, is replaced by
    // zeros when staged, or is never used.
    const int k = min(min(step, steps - 1) * kStep + ld_chunk * 16, K - 16);
    xr[decltype(set)::value][decltype(piece)::value] =
        *reinterpret_cast<const i32x4_unaligned*>(xp[decltype(piece)::value] + k);
  };
  auto store_x_piece = [&](int step, auto set, auto piece) {
    constexpr int p = decltype(piece)::value;
    i32x4 v = xr[decltype(set)::value % kSlots][p];
    if (kRagged) v = ShiftBytesDown(v, step == ragged_step ? ragged_skip : 0);
    if (upper_chunk && step == half_step) v = i32x4{0, 0, 0, 0};
    *reinterpret_cast<i32x4*>(smem + decltype(set)::value % 2 * kStageBytes + st_off +
                              p * 32 * kXStride) = v;
  };
  // Operand of batch tile j, sub-step h: lane L reads row 32 j + L % 32, bytes
  // 32 h + 16 * (L / 32) .. +16 of the staged 128.
  const int frag_off = (lane & 31) * kXStride + (lane >> 5) * 16;
  auto read_frag = [&](auto stage, int j, int h) {
    return *reinterpret_cast<const i32x4*>(smem + decltype(stage)::value * kStageBytes + frag_off +
                                           j * 32 * kXStride + h * 32);
  };
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
  constexpr auto kTiles = std::make_integer_sequence<int, kWaveTiles>{};
  constexpr auto kSubs = std::make_integer_sequence<int, kSub>{};
  constexpr auto kChunks = std::make_integer_sequence<int, kXChunks>{};

  i32x16 acc[kWaveTiles][kBatchTiles];
#pragma unroll
  for (int i = 0; i < kWaveTiles; ++i) {
#pragma unroll
    for (int j = 0; j < kBatchTiles; ++j) {
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;
    }
  }

  // Prologue: rows of steps 0 and 1 staged, those of the steps up to kSlots requested, weights of the
  // first kSlots steps requested, operands of step 0 read.
  ForEachConst(kChunks, [&](auto p) { load_x_piece(0, C0{}, p); });
  ForEachConst(kChunks, [&](auto p) { load_x_piece(1, C1{}, p); });
  asm volatile("" ::: "memory");
  constexpr auto kTurn = std::make_integer_sequence<int, kSlots>{};
  ForEachConst(kTurn, [&](auto slot) {
    ForEachConst(kTiles, [&](auto i) {
      ForEachConst(kSubs, [&](auto h) { load_w_piece(decltype(slot)::value, slot, i, h); });
    });
  });
  asm volatile("" ::: "memory");
  ForEachConst(kChunks, [&](auto p) { store_x_piece(0, C0{}, p); });
  ForEachConst(kChunks, [&](auto p) { store_x_piece(1, C1{}, p); });
  asm volatile("" ::: "memory");
  ForEachConst(std::make_integer_sequence<int, kSlots - 1>{}, [&](auto n) {
    constexpr int kStepAhead = decltype(n)::value + 2;
    ForEachConst(kChunks, [&](auto p) {
      load_x_piece(kStepAhead, std::integral_constant<int, kStepAhead % kSlots>{}, p);
    });
  });
  asm volatile("" ::: "memory");
  if (tid < BN) chan_params[tid] = chan_p;
  // The short requantization (RequantizeShort) needs every channel of the tile to shift right by
  // 1..31 bits and |accumulator + addend| < 2^30, which |addend| < 2^29 and a depth of at most
  // 32768 guarantee; one channel outside that sends the whole workgroup down the general form.
  // The short float epilogue multiplies zero point and row sum as 24-bit integers: |row sum| is at
  // most 128 K.
  const bool general_form =
      EPI == Int8Epilogue::kRequantize
          ? __syncthreads_or((tid < BN && !plain_channel) || K > 32768 || a.act_min > a.act_max)
          : __syncthreads_or((EPI == Int8Epilogue::kHybrid && (!small_zero || K > 65535)) ||
                             a.activation == 5 || a.batch_matmul || zero_input);
  i32x4 fa[kBatchTiles][kSub];
#pragma unroll
  for (int j = 0; j < kBatchTiles; ++j) {
#pragma unroll
    for (int h = 0; h < kSub; ++h) fa[j][h] = read_frag(C0{}, j, h);
  }

  // One depth step s (slot = s % kSlots). MFMA number m works on sub-step h = m / kHalf, channel tile
  // i = (m % kHalf) / kBatchTiles, batch tile j = m % kBatchTiles; what follows it:
  //   * after the first MFMA that frees an operand of the rows: the barrier that publishes the
  //     rows of step s + 1 (staged at the end of step s - 1);
  //   * after the last use of fa[j][h] (i = last tile): its LDS read for step s + 1;
  //   * after the last use of weight piece (i, h) (j = last batch tile): its load for step s + kSlots;
  //   * spread over the step: the loads of the rows of step s + kSlots + 1;
  //   * from the middle of the step on, one every few MFMAs: the LDS writes of the rows of step
  //     s + 2, into the buffer whose readers all passed this step's barrier (behind the last
  //     MFMAs instead they are still in the LDS queue when the next step's barrier waits for
  //     them: 1.6 us per launch of config 4 at the nominal clock).
  // The scheduling fences keep exactly this order. Vector memory returns in issue order, which
  // the waits the compiler derives from the registers respect.
  constexpr int kHalf = kBatchTiles * kWaveTiles;
  constexpr int kMfmas = kSub * kHalf;
  constexpr int kFirstFree = (kWaveTiles - 1) * kBatchTiles;
  constexpr int kStoreAt = kMfmas / 4, kStoreEvery = (kMfmas / 2) / kXChunks;
  auto step_body = [&](int s, auto slot) {
    constexpr int kSlot = decltype(slot)::value;
    using Slot = std::integral_constant<int, kSlot>;
    using Next = std::integral_constant<int, (kSlot + 1) % kSlots>;
    using AfterNext = std::integral_constant<int, kSlot + 2>;
    using Other = std::integral_constant<int, 1 - kSlot % 2>;
    ForEachConst(std::make_integer_sequence<int, kMfmas>{}, [&](auto index) {
      constexpr int m = decltype(index)::value;
      constexpr int h = m / kHalf, i = (m % kHalf) / kBatchTiles, j = m % kBatchTiles;
      acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wring[kSlot][i][h], fa[j][h], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (m == kFirstFree) {
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (i == kWaveTiles - 1) {
        fa[j][h] = read_frag(Other{}, j, h);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (j == kBatchTiles - 1) {
        load_w_piece(s + kSlots, Slot{}, std::integral_constant<int, i>{}, std::integral_constant<int, h>{});
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (m % (kMfmas / kXChunks) == 1) {
        load_x_piece(s + kSlots + 1, Next{}, std::integral_constant<int, m / (kMfmas / kXChunks)>{});
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (m >= kStoreAt && (m - kStoreAt) % kStoreEvery == 0 &&
                    (m - kStoreAt) / kStoreEvery < kXChunks) {
        store_x_piece(s + 2, AfterNext{},
                      std::integral_constant<int, (m - kStoreAt) / kStoreEvery>{});
        __builtin_amdgcn_sched_barrier(0);
      }
    });
  };

  // Whole turns of the slots run without branches so that they stay fixed registers.
  int s0 = 0;
  for (; s0 + kSlots <= steps; s0 += kSlots) {
    ForEachConst(kTurn, [&](auto slot) { step_body(s0 + decltype(slot)::value, slot); });
  }
  ForEachConst(std::make_integer_sequence<int, kSlots - 1>{}, [&](auto slot) {
    if (s0 + decltype(slot)::value < steps) step_body(s0 + decltype(slot)::value, slot);
  });

  // Epilogue. Register e of acc[i][j] holds channel 32 i + 8 * (e / 4) + 4 * (L / 32) + e % 4 of
  // the wavefront's 64 and batch row 32 j + L % 32 of the workgroup's 128: four groups (g) of
  // four consecutive channels per lane and tile.
  const int row_in_tile = lane & 31;
  // The clamp bounds in vector registers: v_med3_i32 takes at most one scalar operand.
  int32_t act_lo = a.act_min, act_hi = a.act_max;
  asm volatile("" : "+v"(act_lo), "+v"(act_hi));
  // The outputs of a tile are put together in LDS (the row buffers, free by now) and leave in
  // 16-byte pieces, neighbouring lanes on neighbouring pieces of a row, i.e. in whole cache
  // lines. Stored from the accumulator layout a store instruction touches 32 rows with 8 bytes
  // each, and the 8 MB of config 4's output reach L2 as a million partial-line writes behind the
  // last MFMA. kFull: an interior tile, no bounds test; tiles at the edge store what lies inside,
  // the last piece of a row value by value. Rows of any length start on any byte (an int8 output
  // of an odd channel count): the pieces' addresses need no alignment.
  constexpr int kOutStride = BN + 16;
  static_assert(BM * kOutStride <= 2 * kStageBytes, "output tile does not fit the row buffers");
  auto epilogue_int8 = [&](auto full_tag, auto short_tag) {
    constexpr bool kFull = decltype(full_tag)::value;
    constexpr bool kShort = decltype(short_tag)::value;
    __syncthreads();  // every wavefront has read its last row operands
#pragma unroll
    for (int i = 0; i < kWaveTiles; ++i) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int local = (wave * kWaveTiles + i) * 32 + 8 * g + 4 * (lane >> 5);
        int32_t mult[4], shift[4], addend[4], half[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const i32x4 p = chan_params[local + r];
          mult[r] = p[0];
          shift[r] = kShort ? -p[1] : p[1];
          addend[r] = p[2];
          half[r] = p[3];
        }
#pragma unroll
        for (int j = 0; j < kBatchTiles; ++j) {
          int32_t q[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            q[r] = kShort ? RequantizeShort(acc[i][j][4 * g + r] + addend[r], mult[r], shift[r],
                                            half[r], a.output_offset, act_lo, act_hi)
                          : RequantizeCore(acc[i][j][4 * g + r] + addend[r], mult[r], shift[r],
                                           a.output_offset, a.act_min, a.act_max);
          }
          *reinterpret_cast<int32_t*>(smem + (j * 32 + row_in_tile) * kOutStride + local) =
              PackLowBytes(q[0], q[1], q[2], q[3]);
        }
      }
    }
    __syncthreads();
    constexpr int kPiecesPerRow = BN / 16;
#pragma unroll
    for (int k = 0; k < BM * kPiecesPerRow / kThreads; ++k) {
      const int piece = k * kThreads + tid;
      const int row = piece / kPiecesPerRow, at = (piece % kPiecesPerRow) * 16;
      const int8_t* from = smem + row * kOutStride + at;
      int8_t* to = a.output_i8 + static_cast<size_t>(m0 + row) * N + n0 + at;
      const int inside = kFull ? 16 : (m0 + row < M ? N - (n0 + at) : 0);
      if (inside >= 16) {
        *reinterpret_cast<i32x4_unaligned*>(to) = *reinterpret_cast<const i32x4*>(from);
      } else {
        for (int b = 0; b < inside; ++b) to[b] = from[b];
      }
    }
  };
  // Float outputs go 32 rows (one batch tile) at a time: a wavefront then stores one row's whole
  // kilobyte per instruction instead of 32 bytes in each of 32 rows.
  // form_tag: 0 the general form; 1 and 2 a FULLY_CONNECTED product without and with a clamp. A
  // wavefront alone on its SIMD issues a vector operation every 8 cycles or so, and the general
  // form's 35 per output (both arithmetics, a 32-bit product at a quarter of the rate, a walk of
  // the activations) for 128 outputs a lane were 10 us of a launch: 512 x 4096 -> 14336 53.8 us
  // with the row quantizer, now 43.7.
  const float clamp_lo = a.activation == 2 ? -1.0f : 0.0f;
  const float clamp_hi =
      a.activation == 2 ? 1.0f : (a.activation == 3 ? 6.0f : __builtin_inff());
  auto epilogue_float = [&](auto full_tag, auto form_tag) {
    constexpr bool kFull = decltype(full_tag)::value;
    constexpr int kForm = decltype(form_tag)::value;
    // ApplyFloatActivation's clamps, one expression for all three.
    auto activate = [&](float v) {
      if (kForm == 0) return ApplyFloatActivation(v, a.activation);
      if (kForm == 1) return v;
      const float t = (clamp_hi < v) ? clamp_hi : v;
      return (clamp_lo < t) ? t : clamp_lo;
    };
    constexpr int kRowBytes = BN * 4 + 16;
    static_assert(32 * kRowBytes <= 2 * kStageBytes, "a batch tile of floats does not fit");
    constexpr int kPiecesPerRow = BN / 4;
    // The lane's channels, read from LDS once for all batch tiles (the registers of the loop's operands
    // are free by now).
    float chan_scale[kWaveTiles][4][4], chan_bias[kWaveTiles][4][4];
    int32_t chan_sum[kWaveTiles][4][4];
#pragma unroll
    for (int i = 0; i < kWaveTiles; ++i) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const i32x4 p = chan_params[(wave * kWaveTiles + i) * 32 + 8 * g + 4 * (lane >> 5) + r];
          chan_scale[i][g][r] = __int_as_float(p[0]);
          chan_bias[i][g][r] = __int_as_float(p[1]);
          chan_sum[i][g][r] = p[2];
        }
      }
    }
#pragma unroll
    for (int j = 0; j < kBatchTiles; ++j) {
      const float bscale = row_scale[j];
      const int32_t bzp = row_zero[j];
      __syncthreads();  // the buffer's last readers (main loop, previous batch tile) are through
#pragma unroll
      for (int i = 0; i < kWaveTiles; ++i) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int local = (wave * kWaveTiles + i) * 32 + 8 * g + 4 * (lane >> 5);
          float v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float scale = chan_scale[i][g][r], bias = chan_bias[i][g][r];
            const int32_t row_sum = chan_sum[i][g][r];
            const int32_t dot = acc[i][j][4 * g + r];
            if (EPI == Int8Epilogue::kHybrid4Bit) {
              v[r] = activate(Hybrid4BitCore(dot, bscale, scale, bzp, bias, a.bias_f32 != nullptr, 0));
            } else if (kForm != 0) {
              v[r] = activate(__fadd_rn(
                  bias, __fmul_rn(static_cast<float>(dot - __mul24(row_sum, bzp)),
                                  __fmul_rn(bscale, scale))));
            } else {
              v[r] = HybridCoreSelect(dot, bscale, scale, bzp, row_sum, bias, a.activation,
                                      a.batch_matmul != 0, zero_input);
            }
          }
          *reinterpret_cast<float4*>(smem + row_in_tile * kRowBytes + local * 4) =
              make_float4(v[0], v[1], v[2], v[3]);
        }
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 32 * kPiecesPerRow / kThreads; ++k) {
        const int piece = k * kThreads + tid;
        const int row = piece / kPiecesPerRow, at = (piece % kPiecesPerRow) * 4;
        const float* from = reinterpret_cast<const float*>(smem + row * kRowBytes) + at;
        float* to = a.output_f32 + static_cast<size_t>(m0 + j * 32 + row) * N + n0 + at;
        const int inside = kFull ? 4 : (m0 + j * 32 + row < M ? N - (n0 + at) : 0);
        if (inside >= 4) {
          *reinterpret_cast<f32x4_unaligned*>(to) = *reinterpret_cast<const f32x4_unaligned*>(from);
        } else {
          for (int c = 0; c < inside; ++c) to[c] = from[c];
        }
      }
    }
  };
  const bool interior = m0 + BM <= M && n0 + BN <= N;
  if (EPI != Int8Epilogue::kRequantize) {
    using General = std::integral_constant<int, 0>;
    using Plain = std::integral_constant<int, 1>;
    using Clamped = std::integral_constant<int, 2>;
    if (general_form) {
      epilogue_float(std::false_type{}, General{});
    } else if (a.activation == 0) {
      if (interior) {
        epilogue_float(std::true_type{}, Plain{});
      } else {
        epilogue_float(std::false_type{}, Plain{});
      }
    } else if (interior) {
      epilogue_float(std::true_type{}, Clamped{});
    } else {
      epilogue_float(std::false_type{}, Clamped{});
    }
  } else if (!general_form) {
    if (interior) {
      epilogue_int8(std::true_type{}, std::true_type{});
    } else {
      epilogue_int8(std::false_type{}, std::true_type{});
    }
  } else {
    epilogue_int8(std::false_type{}, std::false_type{});
  }
}

template <int BM, int kWaveTiles, bool kRagged, int kSlots>
hipError_t LaunchForm(const FcInt8Args& a, Int8Epilogue epilogue, int grid, hipStream_t stream) {
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kThreads), 0, stream, a);
    return hipGetLastError();
  };
  switch (epilogue) {
    case Int8Epilogue::kRequantize:
      return launch(FcInt8PackedGemmKernel<Int8Epilogue::kRequantize, BM, kWaveTiles, kRagged, kSlots>);
    case Int8Epilogue::kHybrid:
      return launch(FcInt8PackedGemmKernel<Int8Epilogue::kHybrid, BM, kWaveTiles, kRagged, kSlots>);
    default:
      return launch(FcInt8PackedGemmKernel<Int8Epilogue::kHybrid4Bit, BM, kWaveTiles, kRagged, kSlots>);
  }
}

template <int BM, int kWaveTiles, int kSlots>
hipError_t LaunchShape(const FcInt8Args& a, Int8Epilogue epilogue, int grid, hipStream_t stream) {
  return a.depth % 16 ? LaunchForm<BM, kWaveTiles, true, kSlots>(a, epilogue, grid, stream)
                      : LaunchForm<BM, kWaveTiles, false, kSlots>(a, epilogue, grid, stream);
}

constexpr int kMinLargeTiles = 128;
constexpr int kCus = 256;

int LargeTiles(const FcInt8Args& a) {
  return ((a.batches + 127) / 128) * ((a.out_depth + 255) / 256);
}
int SquareTiles(const FcInt8Args& a) {
  return ((a.batches + 127) / 128) * ((a.out_depth + 127) / 128);
}
int SmallTiles(const FcInt8Args& a) {
  return ((a.batches + 63) / 64) * ((a.out_depth + 127) / 128);
}

// 64 x 128 tiles, a workgroup at most per CU: a wavefront alone on its SIMD waits out every load that
// it asked for less than a memory latency before, and a step of this tile is 256 matrix-core
// cycles. With two register sets rows had one step to arrive in (a step took 0.42 us); four sets cost
// the second workgroup of a CU nothing where there is none. Two sets -> four, us, filters in the
// cache / from memory: 300 x 4096 -> 4096 15.9 -> 12.9 / 20.3 -> 16.6, 400 x 11008 -> 4096 37.2 -> 29.5
// / 49.6 -> 38.4, 256 x 8192 -> 6144 27.8 -> 23.0 / 40.0 -> 32.5, 300 x 3072 -> 5120 13.6 -> 12.2 /
// 17.2 -> 14.7. A short walk gains only on filters from memory (400 x 2048 -> 4096 8.0 -> 8.5 /
// 10.1 -> 9.1, 400 x 512 -> 4096 5.2 -> 5.4 / 5.9 -> 6.0), and in more than one workgroup per CU they
// hide each other's waits (300 x 8192 -> 8192, 320 workgroups, 39.7 -> 44.0).
bool DeepRing(const FcInt8Args& a) { return a.depth > 2048 && SmallTiles(a) <= kCus; }

// Of the launches on smaller tiles: 128 x 128 moves two thirds of the bytes per product that 64 x 128
// does. Among those that 128 x 256 would give half the chip or more, all but the short walks in one
// round (see FcInt8PackedGemmForm). Below, where it makes one round of what 64 x 128 takes more than one
// for (us, 64 x 128 -> 128 x 128, filters in the cache / from memory): 350 x 7792 -> 6425 50.6 -> 35.6
// / 50.1 -> 47.6, 494 x 7376 -> 4530 36.5 -> 30.7 / 48.8 -> 43.5, 256 x 4096 -> 14336 22.8 -> 21.6 / 30.8
// -> 28.1; least 1110 x 2240 -> 2805 14.9 -> 14.0 / 15.9 -> 15.3. (Shorter walks: 819 x 1392 -> 4231
// 11.3 -> 12.2.) Of 370 such sizes with 156 tiles and more it takes 0.90 / 0.93 of the time of 64 x 128, float
// outputs 0.94 / 0.97; of 100 with fewer 0.89 / 1.04 and 0.93 / 1.08 (640 x 7256 -> 3511, 140 tiles: 41.5 ->
// 39.8 / 40.7 -> 45.6): half the CUs ask for the whole filter.
bool TakesSquareTiles(const FcInt8Args& a) {
  if (LargeTiles(a) >= kMinLargeTiles) return LargeTiles(a) > kCus || a.depth > 2048;
  return a.depth >= 2048 && SmallTiles(a) > kCus && SquareTiles(a) <= kCus;
}

}  // namespace

bool FcInt8PackedGemmSupports(const FcInt8Args& a) {
  return a.depth >= 16 && a.filter_offset == 0 && a.batches > 0 && a.out_depth > 0 &&
         (reinterpret_cast<uintptr_t>(a.filter) & 15) == 0;
}

// 128 x 256 tiles move the fewest bytes per MFMA; a launch they would cut into fewer workgroups than
// half the chip's CUs takes smaller tiles instead, or, where those leave it idle too, small tiles
// with the depth split over the wavefronts. Above that line smaller tiles win where the walk is
// short, because of a large tile's prologue and epilogue (9 us of a workgroup's time, and no second
// workgroup on its CU to hide them), and where large tiles make exactly half a round.
// (us, 128 x 256 -> chosen, filters in the cache / from memory:)
//   more than a round, depth 512 to 2048, to 128 x 128: 2048 x 1024 -> 14336 52.6 -> 47.5 / 57.5 -> 51.5,
//     700 x 1024 -> 14336 24.7 -> 20.8 / 27.7 -> 23.3, 1715 x 560 -> 15924 52.4 -> 41.9 / 53.1 -> 42.3. Float
//     outputs gain more: hybrid 2048 x 1024 -> 14336 76 -> 63 / 83 -> 73. Of 220 such sizes where they fill
//     less than two rounds for one of 128 x 256 0.85 of the time in the mean (least 1.03), of 100 where they
//     fill two 0.96 (least 1.04). Rows that end inside a 16-byte piece are read twice as often from addresses
//     that are no multiple of 16: deeper than 1024 and in two rounds for one they lose (1.05 of the time in
//     the mean, 1778 x 1949 -> 6928 46.9 -> 60 / 44.5 -> 53, 1600 x 1434 -> 7948 38.6 -> 46 / 38.2 -> 42) and stay.
//   a round at most, depth 512 to 768, to 64 x 128 as long as those are three rounds: 1506 x 672 -> 2567 13.8 ->
//     8.5 / 14.5 -> 9.2, 1806 x 608 -> 2575 13.4 -> 10.5 / 14.2 -> 11.3; of 66 such sizes 0.86 of the time in the
//     mean, least 1.01. (In a fourth round: 392 x 704 -> 14656 14.3 -> 17.7 / 13.2 -> 17.1, 652 x 576 -> 9024
//     12.4 -> 15.9 / 12.0 -> 14.3. Deeper: 750 x 912 -> 8538 16.5 -> 20.8.)
//   half a round, depth above 2048, to one round of 128 x 128: 1000 x 4096 -> 4096 26.0 -> 22.4 / 30.2 -> 25.3; 17
//     sizes, least 0.83 of the time.
// Shallower launches than 512 are not in those figures and stay.
Int8GemmForm FcInt8PackedGemmForm(const FcInt8Args& a) {
  const int large = LargeTiles(a);
  if (large >= kMinLargeTiles) {
    const int square = SquareTiles(a);
    const auto rounds = [](int tiles) { return (tiles + kCus - 1) / kCus; };
    const bool two_for_one = rounds(square) >= 2 * rounds(large);
    const bool smaller = large > kCus ? a.depth >= 512 && a.depth <= 2048 &&
                                            !(a.depth % 16 && a.depth > 1024 && two_for_one)
                                      : (a.depth >= 512 && a.depth <= 768 && SmallTiles(a) <= 3 * kCus) ||
                                            (a.depth > 2048 && square <= kCus);
    if (!smaller) return Int8GemmForm::kTiles128x256;
  } else if (FcInt8SplitGemmBeatsTiles(a, SmallTiles(a))) {
    return Int8GemmForm::kSplit;
  }
  if (TakesSquareTiles(a)) return Int8GemmForm::kTiles128x128;
  return DeepRing(a) ? Int8GemmForm::kTiles64x128Ahead : Int8GemmForm::kTiles64x128;
}

// A few tiles more than one per CU cost a second round, nearly all of it on an idle chip. The rows of that
// tail go in a launch of their own then, on the tiles that suit them: the number of rows the first
// launch keeps. For tails up to a quarter of a round and walks deeper than 2048 (shorter ones are on
// smaller tiles), us, one launch -> two: 2048 x 7808 -> 4352, 272 tiles, 103 -> 84-92; 2048 x 4096 -> 4352
// 59.4 -> 50.8; 1100 x 4096 -> 8192, 288 tiles, 60.8 -> 50.2; 1800 x 4096 -> 5120, 300 tiles, 58.9 -> 50.2;
// least 1614 x 5680 -> 5909, 312 tiles, 83 -> 81. A larger tail gains less (800 x 4096 -> 12288, 336
// tiles, 61.8 -> 59.6), one behind two or three rounds loses (2048 x 4096 -> 8448 96.6 -> 104, 2048 x 2560 ->
// 12800 93 -> 107: the last tiles of a round overlap the first of the next).
int FcInt8PackedGemmFirstRows(const FcInt8Args& a) {
  const int tiles = LargeTiles(a);
  if (a.depth <= 2048 || tiles <= kCus || tiles > kCus + kCus / 4) return a.batches;
  const int tiles_n = (a.out_depth + 255) / 256;
  const int kept = kCus / tiles_n;  // rows of tiles
  if (kept * tiles_n < kCus - kCus / 16) return a.batches;
  return min(kept * 128, a.batches);
}

hipError_t LaunchFcInt8PackedGemm(const FcInt8Args& a, Int8Epilogue epilogue, hipStream_t stream) {
  if (!FcInt8PackedGemmSupports(a)) return hipErrorNotSupported;
  if (const int kept = FcInt8PackedGemmFirstRows(a); kept < a.batches) {
    FcInt8Args part = a;
    part.whole_input = a.whole_input ? a.whole_input : a.input;
    part.whole_batches = a.whole_input ? a.whole_batches : a.batches;
    part.batches = kept;
    if (hipError_t err = LaunchShape<128, 2, 2>(part, epilogue, LargeTiles(part), stream)) return err;
    const size_t rows = kept, out = rows * a.out_depth;
    part.batches = a.batches - kept;
    part.input += rows * a.depth;
    if (part.output_i8) part.output_i8 += out;
    if (part.output_f32) part.output_f32 += out;
    if (part.scaling_factors) part.scaling_factors += rows;
    if (part.zero_points) part.zero_points += rows;
    return LaunchFcInt8PackedGemm(part, epilogue, stream);
  }
  switch (FcInt8PackedGemmForm(a)) {
    case Int8GemmForm::kSplit: return LaunchFcInt8SplitGemm(a, epilogue, stream);
    case Int8GemmForm::kTiles64x128: return LaunchShape<64, 1, 2>(a, epilogue, SmallTiles(a), stream);
    case Int8GemmForm::kTiles64x128Ahead: return LaunchShape<64, 1, 4>(a, epilogue, SmallTiles(a), stream);
    case Int8GemmForm::kTiles128x128: return LaunchShape<128, 1, 2>(a, epilogue, SquareTiles(a), stream);
    case Int8GemmForm::kTiles128x256: return LaunchShape<128, 2, 2>(a, epilogue, LargeTiles(a), stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace lrtfc
