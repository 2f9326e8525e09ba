// FULLY_CONNECTED on the re-tiled int8 filter for the sizes between decode and prefill: batches of
// tens to hundreds of rows against filters that 128 x 256 tiles would cut into too few workgroups
// to fill the chip.
//
//   out[m, n] = epilogue(sum_k x[m, k] * w[n, k])        x [M, K] row-major int8
//
// Such a launch is bound by latency: with the whole depth walked by one wavefront per SIMD (the
// GEMM of the large tiles) every 128 deep step costs a memory latency, about 1270 cycles of which
// 256 are matrix work. Here a workgroup is eight wavefronts on ONE small output tile, and the
// depth is dealt to them in steps of 128: no barrier until the end, both operands requested by the
// wavefront that multiplies them one step ahead of itself, so a CU has its 64 KB of outstanding
// loads filled by independent wavefronts. The eight int32 partial tiles meet in LDS by integer atomics (exact in any order).
//
// Small tiles move more bytes per product: a 64 x 64 tile reads 128 bytes per 4096 products, which
// at 64 bytes per clock and CU bounds the matrix cores to half their rate; the rule that picks the
// tile (Cost) weighs that against the rounds of workgroups. Measured: 77 x 2999 -> 5003 12.2 ->
// 7.1 us, 100 x 16384 -> 512 30.2 -> 10.0 us, 200 x 4096 -> 4096 11.6 -> 9.6 us.
#include "fc_epilogues.h"
#include "kernels.h"

namespace lrtfc {
namespace {

using i32x16 = int __attribute__((ext_vector_type(16)));

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;
constexpr int kSlab = 64;   // depth of one tile of the packed filter
constexpr int kStep = 128;  // depth per step of a wavefront: two slabs, one cache line of a row
constexpr int kSub = kStep / 32;
constexpr int kRowStride = kStep + 16;  // of a staged row: operand reads without bank conflicts

// Lanes of one wavefront exchange rows through LDS, whose operations the hardware keeps in the
// wavefront's order: only the compiler has to be kept from moving them past each other.
__device__ __forceinline__ void LaneFence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
}

// RT x CT tiles of 32 rows x 32 channels per workgroup.
template <Int8Epilogue EPI, int RT, int CT>
__global__ __launch_bounds__(kThreads, RT * CT == 4 ? 2 : 4)
void FcInt8SplitGemmKernel(FcInt8Args a, int tiles, bool rows_inner, int total, int per_xcd) {
  constexpr int BM = RT * 32, BN = CT * 32;
  constexpr int kSumStride = BN + 1;  // 32 rows at one channel lie in 32 banks
  __shared__ __align__(16) int8_t rows[kWaves * BM * kRowStride];
  __shared__ int32_t sums[BM * kSumStride];
  __shared__ int32_t row_scale[BM], row_zero[BM];  // float bits; zero points
  const int M = a.batches, N = a.out_depth, K = a.depth;
  const int slabs = (K + kSlab - 1) / kSlab;
  const int steps = (slabs + 1) / 2;

  // Workgroups are dealt round-robin to the 8 XCDs; each takes a contiguous range of tiles. With the
  // row tiles of one channel range next to each other (rows_inner) a filter tile is fetched into one
  // L2 once, and every L2 fetches the rows; where those are the larger operand it is the other way
  // round (2048 x 3072 -> 512 8.6 us, rows inner 12.8; 1500 x 16384 -> 1024 52 and 57).
  const int id = static_cast<int>(blockIdx.x % 8) * per_xcd + static_cast<int>(blockIdx.x / 8);
  if (static_cast<int>(blockIdx.x / 8) >= per_xcd || id >= total) return;
  const int inner = id % tiles, outer = id / tiles;
  const int m0 = (rows_inner ? inner : outer) * BM, n0 = (rows_inner ? outer : inner) * BN;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // Operands: lane L holds 16 depth bytes of half L / 32 of a 32-deep sub-step for channel (row)
  // L % 32 of a tile. Indices past the edge are clamped: duplicates, computed and not stored.
  const int ctiles = (N + 15) / 16;
  const int half = lane >> 5;
  const int8_t* wp[CT];
#pragma unroll
  for (int i = 0; i < CT; ++i) {
    const int ct = min(n0 / 16 + i * 2 + ((lane & 31) >> 4), ctiles - 1);
    wp[i] = a.filter + static_cast<size_t>(ct) * slabs * 1024 + (lane & 15) * 16 + half * 256;
  }
  // Rows: eight lanes read one whole cache line of a row (its step), 8 rows per instruction. Read in
  // the operands' own layout instead, 32 bytes of 32 rows, the loads are bound by their 32 cache
  // lines each (1.9x the time at 64 rows of 4096). The lines pass through LDS of the wavefront's
  // own: no barrier, its LDS operations keep their order.
  const int piece = lane & 7;
  const int8_t* xp[RT][4];
#pragma unroll
  for (int j = 0; j < RT; ++j) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      xp[j][p] = a.input + static_cast<size_t>(min(m0 + 32 * j + 8 * p + (lane >> 3), M - 1)) * K;
    }
  }
  int8_t* const stage = rows + wave * (BM * kRowStride);
  int8_t* const stage_to = stage + (lane >> 3) * kRowStride + piece * 16;
  const int8_t* const stage_from = stage + (lane & 31) * kRowStride + half * 16;
  i32x4 w[CT][kSub], xr[RT][4], x[RT][kSub];
  // Behind the end of a row (the last step) the addresses are clamped into it: what they read
  // meets zero weights, or is not multiplied at all (a slab that the filter does not have).
  auto load_rows = [&](int step) {
    const int at = min(step * kStep + piece * 16, K - 16);
#pragma unroll
    for (int j = 0; j < RT; ++j) {
#pragma unroll
      for (int p = 0; p < 4; ++p) xr[j][p] = *reinterpret_cast<const i32x4_unaligned*>(xp[j][p] + at);
    }
  };
  auto load_weights = [&](int step, int h) {
    const int slab = min(2 * step + h / 2, slabs - 1);
#pragma unroll
    for (int i = 0; i < CT; ++i) {
      w[i][h] = *reinterpret_cast<const i32x4*>(wp[i] + static_cast<size_t>(slab) * 1024 + (h & 1) * 512);
    }
  };
  auto stage_rows = [&] {
#pragma unroll
    for (int j = 0; j < RT; ++j) {
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        *reinterpret_cast<i32x4*>(stage_to + (32 * j + 8 * p) * kRowStride) = xr[j][p];
      }
    }
  };
  auto read_operands = [&] {
#pragma unroll
    for (int h = 0; h < kSub; ++h) {
#pragma unroll
      for (int j = 0; j < RT; ++j) {
        x[j][h] = *reinterpret_cast<const i32x4*>(stage_from + 32 * j * kRowStride + h * 32);
      }
    }
  };
  // Epilogue inputs: this thread's channel, and for the threads below BM one row of the tile. Requested
  // ahead of the operands, so that nothing at the end waits for memory.
  const int local_n = tid % BN;
  const int n = min(n0 + local_n, N - 1);
  int32_t p0, p1, p2 = 0, row_s = 0, row_z = 0;
  if (EPI == Int8Epilogue::kRequantize) {
    p0 = a.per_channel ? a.multipliers[n] : a.multipliers[0];
    p1 = a.per_channel ? a.shifts[n] : a.shifts[0];
    p2 = a.bias_i32 ? a.bias_i32[n] : 0;
    if (a.input_offset != 0) p2 += a.input_offset * a.filter_row_sums[n];
  } else {
    p0 = __float_as_int(a.per_channel_scales ? a.per_channel_scales[n] : a.filter_scale);
    p1 = __float_as_int(a.bias_f32 ? a.bias_f32[n] : 0.0f);
    if (EPI == Int8Epilogue::kHybrid && a.zero_points) p2 = a.filter_row_sums[n];
    const int m = min(m0 + tid, M - 1);
    row_s = __float_as_int(a.scaling_factors[m]);
    row_z = a.zero_points ? a.zero_points[m] : 0;
  }
  if (wave < steps) {
    load_rows(wave);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int h = 0; h < kSub; ++h) load_weights(wave, h);
  }
  __builtin_amdgcn_sched_barrier(0);

  // EvalHybridDense's early exit for a whole-zero input matters only where a bias element is
  // -0.0f: a workgroup with such a channel settles the question here.
  bool zero_input = false;
  if (EPI == Int8Epilogue::kHybrid && a.zero_input_exit && a.bias_f32 != nullptr) {
    if (__syncthreads_or(n0 + local_n < N && IsNegativeZero(__int_as_float(p1)))) {
      zero_input = a.whole_input
                       ? WorkgroupAllZeroInt8(a.whole_input, static_cast<size_t>(a.whole_batches) * K)
                       : WorkgroupAllZeroInt8(a.input, static_cast<size_t>(M) * K);
    }
  }
  for (int i = tid; i < BM * kSumStride; i += kThreads) sums[i] = 0;
  if (EPI != Int8Epilogue::kRequantize && tid < BM) {
    row_scale[tid] = row_s;
    row_zero[tid] = row_z;
  }
  __syncthreads();

  i32x16 acc[CT][RT];
#pragma unroll
  for (int i = 0; i < CT; ++i) {
#pragma unroll
    for (int j = 0; j < RT; ++j) {
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;
    }
  }
  auto multiply_sub = [&](int h) {
#pragma unroll
    for (int i = 0; i < CT; ++i) {
#pragma unroll
      for (int j = 0; j < RT; ++j) {
        acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[i][h], x[j][h], acc[i][j], 0, 0, 0);
      }
    }
  };
  int step = wave;
  for (; step + kWaves < steps; step += kWaves) {
    stage_rows();
    LaneFence();
    load_rows(step + kWaves);
    __builtin_amdgcn_sched_barrier(0);
    read_operands();
    LaneFence();
#pragma unroll
    for (int h = 0; h < kSub; ++h) {
      multiply_sub(h);
      __builtin_amdgcn_sched_barrier(0);
      load_weights(step + kWaves, h);  // into the registers just read
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (step < steps) {
    if ((K & 15) && step == steps - 1) {  // the row ends inside a piece of this step
      const int skip = RowPieceSkip(step * kStep + piece * 16, K);
#pragma unroll
      for (int j = 0; j < RT; ++j) {
#pragma unroll
        for (int p = 0; p < 4; ++p) xr[j][p] = ShiftBytesDown(xr[j][p], skip);
      }
    }
    stage_rows();
    LaneFence();
    read_operands();
    multiply_sub(0);
    multiply_sub(1);
    if (2 * step + 1 < slabs) {
      multiply_sub(2);
      multiply_sub(3);
    }
    // Register e of acc[i][j]: channel 32 i + 8 (e / 4) + 4 (L / 32) + e % 4, row 32 j + L % 32.
#pragma unroll
    for (int i = 0; i < CT; ++i) {
#pragma unroll
      for (int j = 0; j < RT; ++j) {
        int32_t* to = sums + (32 * j + (lane & 31)) * kSumStride + 32 * i + 4 * half;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          __hip_atomic_fetch_add(to + 8 * (e / 4) + e % 4, acc[i][j][e], __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_WORKGROUP);
        }
      }
    }
  }
  __syncthreads();

  // Neighbouring lanes on neighbouring channels: whole 128- or 256-byte runs of a row per store.
  constexpr int kRowsPerPass = kThreads / BN;
#pragma unroll
  for (int k = 0; k < BM / kRowsPerPass; ++k) {
    const int r = k * kRowsPerPass + tid / BN;
    const int32_t dot = sums[r * kSumStride + local_n];
    if (m0 + r < M && n0 + local_n < N) {
      const size_t at = static_cast<size_t>(m0 + r) * N + n0 + local_n;
      if (EPI == Int8Epilogue::kRequantize) {
        a.output_i8[at] = RequantizeCore(dot + p2, p0, p1, a.output_offset, a.act_min, a.act_max);
      } else if (EPI == Int8Epilogue::kHybrid4Bit) {
        a.output_f32[at] =
            Hybrid4BitCore(dot, __int_as_float(row_scale[r]), __int_as_float(p0), row_zero[r],
                           __int_as_float(p1), a.bias_f32 != nullptr, a.activation);
      } else {
        a.output_f32[at] = HybridCoreSelect(dot, __int_as_float(row_scale[r]), __int_as_float(p0),
                                            row_zero[r], p2, __int_as_float(p1), a.activation,
                                            a.batch_matmul != 0, zero_input);
      }
    }
  }
}

template <int RT, int CT>
hipError_t LaunchTile(const FcInt8Args& a, Int8Epilogue epilogue, hipStream_t stream) {
  const int tiles_m = (a.batches + 32 * RT - 1) / (32 * RT);
  const int tiles_n = (a.out_depth + 32 * CT - 1) / (32 * CT);
  const int total = tiles_m * tiles_n;
  const bool rows_inner = a.batches <= a.out_depth;
  const int inner_tiles = rows_inner ? tiles_m : tiles_n;
  const int per_xcd = (total + 7) / 8;
  const dim3 grid(per_xcd * 8), block(kThreads);
  if (epilogue == Int8Epilogue::kRequantize) {
    hipLaunchKernelGGL((FcInt8SplitGemmKernel<Int8Epilogue::kRequantize, RT, CT>), grid, block, 0,
                       stream, a, inner_tiles, rows_inner, total, per_xcd);
  } else if (epilogue == Int8Epilogue::kHybrid) {
    hipLaunchKernelGGL((FcInt8SplitGemmKernel<Int8Epilogue::kHybrid, RT, CT>), grid, block, 0,
                       stream, a, inner_tiles, rows_inner, total, per_xcd);
  } else {
    hipLaunchKernelGGL((FcInt8SplitGemmKernel<Int8Epilogue::kHybrid4Bit, RT, CT>), grid, block, 0,
                       stream, a, inner_tiles, rows_inner, total, per_xcd);
  }
  return hipGetLastError();
}

// The three tiles. A launch costs about rounds x (fixed + bytes read per workgroup), in bytes at the
// 150 per nanosecond that a CU reaches here; `fixed` (prologue, the join of the eight partial
// tiles, epilogue) was fitted with it to 60 sizes between 24 x 1024 -> 1024 and
// 2000 x 16384 -> 512, where the fit orders the tiles as the measurement does but for near ties.
struct Tile {
  int rows, channels;
  long fixed;
};
constexpr Tile kTiles[] = {{32, 32, 105000}, {32, 64, 180000}, {64, 64, 375000}};
constexpr int kCus = 256;

long Workgroups(const Tile& t, const FcInt8Args& a) {
  return (static_cast<long>(a.batches) + t.rows - 1) / t.rows *
         ((static_cast<long>(a.out_depth) + t.channels - 1) / t.channels);
}

long Cost(const Tile& t, const FcInt8Args& a) {
  return (Workgroups(t, a) + kCus - 1) / kCus *
         (t.fixed + static_cast<long>(t.rows + t.channels) * a.depth);
}

int BestTile(const FcInt8Args& a) {
  int best = 0;
  for (int i = 1; i < 3; ++i) {
    if (Cost(kTiles[i], a) < Cost(kTiles[best], a)) best = i;
  }
  return best;
}

}  // namespace

// Against the kernels that take up to 128 rows in one pass over the filter (int8 rows in,
// microseconds there -> here; "cold": filters rotated through 700 MB, else the same one again).
// Up to 16 rows the register-resident GEMV requests a wavefront's whole share of the filter at once,
// where a wavefront here has one step ahead: on cold filters that weighs more than what these tiles
// save. So the GEMV keeps
//   - rows of at most 16 KB together (9 x 1024 -> 2048 3.6 -> 3.6, cold 3.2 -> 4.0),
//   - shares of more than 24 of its 32 tiles, i.e. depths from 6145 to 8192 (8 x 8192 -> 256
//     5.8 -> 6.3, cold 6.1 -> 8.7),
// unless the tiles make 192 workgroups or more (8 x 4096 -> 6144 7.3 -> 4.8, cold 7.8 -> 7.4). Its rows
// have to fit 64 KB; others, and depths beyond 8192, walk its refilled ring and gain here
// (16 x 8192 -> 1024 11.4 -> 6.5, cold 11.1 -> 9.7). What is left gains on a filter in the cache about
// what it loses on a cold one (16 x 2048 -> 2048 4.8 -> 3.9, cold 4.4 -> 4.8; 12 x 3072 -> 1024
// 5.2 -> 4.3, cold 4.7 -> 5.5; 16 x 4096 -> 1024 5.5 -> 4.7, cold 4.9 -> 6.4).
// Beyond 16 rows: whatever fits one round of small tiles (32 x 2048 -> 2048 6.7 -> 4.5,
// 20 x 2048 -> 16384 9.9 -> 9.0, 48 x 4096 -> 14336 16.5 -> 15.1, 48 x 2048 -> 16384 12.4 -> 9.9);
// the others keep what fills the chip by channel tiles alone (20 x 4096 -> 14336 13.7 -> 13.9,
// 72 rows 19.2 -> 20.6).
bool FcInt8SplitGemmBeatsOnePass(const FcInt8Args& a) {
  // What the GEMM launches for the size is what the figures above are of.
  if (!FcInt8PackedGemmSupports(a) || FcInt8PackedGemmForm(a) != Int8GemmForm::kSplit) return false;
  if (a.batches <= 16) {
    const long tiles = Workgroups(kTiles[0], a);
    if (a.batches < 5 || tiles > kCus) return false;
    const long image = static_cast<long>(a.batches) * ((a.depth + kSlab - 1) / kSlab * kSlab);
    if (image > 65536 || a.depth > 8192) return true;
    if (tiles >= 192) return a.depth > (a.batches < 9 ? 2048 : 1024);
    return image > 16384 && a.depth <= 6144;
  }
  if (a.batches <= 32) {
    return Workgroups(kTiles[a.depth <= 2048 ? 1 : 0], a) <= kCus;
  }
  return a.batches <= 128 && Workgroups(kTiles[2], a) <= kCus;
}

// Against the GEMM on 64 x 128 tiles, in the same unit: 1 us and 0.25 us per 128 deep step and
// round (77 x 2999 -> 5003 12.2 -> 7.1 us, 250 x 2048 -> 2048 9.2 -> 6.1 us, 400 x 8192 -> 2048
// 27.6 -> 15.8 us; 400 x 2048 -> 4096 stays there: 8.1, here 11.4 us).
// What fits one round of tiles is faster here at all 640 sizes measured, or equal (64 x 64 tiles of
// a depth about 1024: 64 x 1024 -> 16384 7.7 us for 8.7, 256 x 1024 -> 4096 1 % slower).
// 64 x 64 tiles in three rounds and more keep all CUs at the L2 at once, which then gives each a third
// of the 150 bytes per nanosecond: at all 66 measured sizes that Cost sends there they are the
// slower ones, by 3 to 37 % (us, 64 x 128 tiles / here: 256 x 4096 -> 10240 20.3 / 27.5,
// 400 x 6144 -> 5120 27.5 / 33.9, 640 x 16384 -> 6144 80 / 103).
bool FcInt8SplitGemmBeatsTiles(const FcInt8Args& a, long workgroups_64x128) {
  const long theirs = (workgroups_64x128 + kCus - 1) / kCus *
                      (150000 + 37500 * ((static_cast<long>(a.depth) + kStep - 1) / kStep));
  const Tile& tile = kTiles[BestTile(a)];
  if (Workgroups(tile, a) <= kCus) return true;
  if (tile.rows * tile.channels == 64 * 64 && Workgroups(tile, a) > 2 * kCus) return false;
  return Cost(tile, a) < theirs;
}

hipError_t LaunchFcInt8SplitGemm(const FcInt8Args& a, Int8Epilogue epilogue, hipStream_t stream) {
  if (!FcInt8PackedGemmSupports(a)) return hipErrorNotSupported;
  switch (BestTile(a)) {
    case 0: return LaunchTile<1, 1>(a, epilogue, stream);
    case 1: return LaunchTile<1, 2>(a, epilogue, stream);
    default: return LaunchTile<2, 2>(a, epilogue, stream);
  }
}

}  // namespace lrtfc
