// Blockwise-int4 FULLY_CONNECTED for prefill batches on gfx950: EvalBlockwise4Bit
// (tflite/kernels/fully_connected.cc:1014-1086) as a matrix-core GEMM.
//
// The decode kernel (fc_int4_packed.hip) streams the whole filter once per four batch rows,
// which is right for one to a few rows and hopeless for hundreds. Here every (row, channel)
// output keeps its float32 accumulator in a register and walks the blocks of 32 depth
// positions in order: one v_mfma_i32_16x16x32_i8 per block and 16 x 16 tile gives the exact
// int32 block sums (its K is exactly one block), and `float(sum) * scale[channel][block]` is
// added to the accumulator unfused, the reference's own order of float operations (:1069-1077),
// so the results are bit-identical to the decode kernel's and the oracle's.
//
// The vector operations per output and block take longer than the matrix cores, and their time adds to the
// MFMAs' (of a block and 16 x 16 tile: 16 cycles of its SIMD, and three operations on its 4 outputs per
// lane 27 from two wavefronts on). Two suffice:
//   * The accumulator input of every MFMA is the bit pattern of 1.5 * 2^23, so its integer result
//     READ AS A FLOAT is 1.5 * 2^23 + sum, exactly (|sum| <= 32 * 8 * 128 < 2^22): no conversion.
//   * fma(that, scale, -1.5 * 2^23 * scale) rounds the exact product sum * scale once, which is
//     what converting and multiplying gives: 1.5 * 2^23 * scale is exact in float32 for a scale
//     of eleven significant bits.
//   * The batch rows are the A operand and the channels the B operand, so that a lane's four results
//     are four rows of ONE channel: one scale per lane and block (and its product with -1.5 * 2^23)
//     serves every row tile, where four channels per lane took four broadcasts per block.
// Bound by issue, at the clock that the power cap leaves: 2048 x 4096 -> 14336 is 3584 tiles of 32 x 32 and
// blocks a SIMD, each 32 cycles of MFMA and 72 of vector operations, 107 for both: 383 thousand cycles, 159 us
// at 2.4 GHz, 193 at the 1.98 GHz that this loop holds on random bits. The launch takes 544 thousand (259 us
// at 2.1 GHz; on constant operands 529 at 2.39), 480 thousand without operand loads, of which the last
// half round of workgroups is 25.
//
// Layouts, made once at prepare (filter) or per call (activations):
//   filter `tile32x32s`: for channel tile t (32 channels) and block b, 1 KiB: lane L's 16 bytes are
//     channel 32 t + L % 32, depths 16 (L / 32) ... + 16 of the block, sign-extended to int8: an
//     operand of v_mfma_i32_32x32x32_i8. After all tiles, the block scales as float32, 32 channels x
//     4 blocks per tile and quad of blocks: a lane's 16-byte load is its channel's scales of four
//     blocks.
//   activations: batch rows in place of channels, either in the same form (`tile32x32`) or, for the
//     small forms, `tile16x64`: 16 rows and a pair of blocks in 1 KiB, lane L's 16 bytes row L % 16,
//     depths 8 (L / 16) ... + 8 of the first block, then of the second. The row quantizer writes
//     either order itself.
// No LDS: a wavefront owns a few tiles and requests the operands of the next blocks while it works
// on the current ones (a ring in registers); both operands are re-read by other wavefronts from L1
// and L2. Two kernels: FcInt4BlockwiseGemmLargeKernel on 32 x 32 tiles, whose one MFMA per block and
// tile does four times the work of a 16 x 16 one in twice the time; and FcInt4BlockwiseGemmKernel on
// 16 x 16 tiles for launches that the large tiles would cut into too few wavefronts.
#include <mutex>

#include "kernels.h"
#include "quantize_device.h"

namespace lrtfc {
namespace {

#define LRTFC_GLOBAL __attribute__((address_space(1)))

constexpr int kThreads = 256;
constexpr int kBlock = 32;    // depth positions per quantization block
constexpr int kTile = 16;     // channels / rows per MFMA tile

using i64 = long;
typedef long i64x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ int SignedNibble(uint32_t byte, int high) {
  const int n = high ? (byte >> 4) : (byte & 0xF);
  return (n ^ 8) - 8;
}

constexpr int kWide = 32;  // channels / rows per tile of the large form

// Model layout (rows of depth / 2 bytes, low nibble = even depth; fp16 scales [N, nb]) ->
// tile32x32s + float32 scales. One thread per 8-byte half of a lane slot of the tile array.
__global__ __launch_bounds__(kThreads) void PackInt4BlockwiseGemmKernel(
    const uint8_t* __restrict__ filter, const uint16_t* __restrict__ scales_f16, int out_depth,
    int depth, int tiles, int nb, uint8_t* __restrict__ dst) {
  const int64_t slot = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  const int quads = (nb + 3) / 4;
  const int64_t slots = static_cast<int64_t>(tiles) * nb * 128;
  if (slot < slots) {
    const int lane = static_cast<int>((slot >> 1) & 63);
    const int64_t tb = slot >> 7;
    const int b = static_cast<int>(tb % nb);
    const int t = static_cast<int>(tb / nb);
    const int n = t * kWide + (lane & 31);
    const int k0 = b * kBlock + 16 * (lane >> 5) + 8 * static_cast<int>(slot & 1);
    uint32_t lo = 0, hi = 0;
    if (n < out_depth) {
      const uint8_t* src = filter + static_cast<size_t>(n) * (depth / 2) + k0 / 2;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t byte = src[j];
        const uint32_t pair = (static_cast<uint32_t>(SignedNibble(byte, 0)) & 0xFF) |
                              (static_cast<uint32_t>(SignedNibble(byte, 1)) & 0xFF) << 8;
        if (j < 2) {
          lo |= pair << (16 * j);
        } else {
          hi |= pair << (16 * (j - 2));
        }
      }
    }
    reinterpret_cast<uint2*>(dst)[slot] = make_uint2(lo, hi);
  }
  // scales: one thread per (tile, quad of blocks, channel, block)
  const int64_t scale_slots = static_cast<int64_t>(tiles) * quads * (kWide * 4);
  if (slot < scale_slots) {
    const int c = static_cast<int>((slot >> 2) & 31);
    const int64_t tq = slot >> 7;
    const int b = 4 * static_cast<int>(tq % quads) + static_cast<int>(slot & 3);
    const int t = static_cast<int>(tq / quads);
    const int n = t * kWide + c;
    float* out = reinterpret_cast<float*>(dst + slots * 8);
    out[slot] = n < out_depth && b < nb
                    ? HalfBitsToFloatFast(scales_f16[static_cast<size_t>(n) * nb + b]) : 0.0f;
  }
}

// Element k of batch row m within its row tile of the tile16x64 layout, as a byte offset
// from the tile row's base.
struct Tile16x64Placement {
  int row_in_tile;
  __device__ __forceinline__ size_t operator()(int k) const {
    const size_t lane_slot = static_cast<size_t>(k >> 6) * 64 + ((k & 31) >> 3) * 16 + row_in_tile;
    return (lane_slot * 2 + ((k >> 5) & 1)) * 8 + (k & 7);
  }
};

// The same within a tile of 32 rows of the tile32x32 layout.
struct Tile32x32Placement {
  int row_in_tile;
  __device__ __forceinline__ size_t operator()(int k) const {
    return static_cast<size_t>(k >> 5) * 1024 + ((k & 31) >> 4) * 512 + row_in_tile * 16 + (k & 15);
  }
};

// BatchQuantizeFloats of float rows [batches, depth] straight into tiles of ROWS rows: one workgroup
// per row of the padded batch (rows past the batch are zero). `tile_bytes`: one row tile.
template <int VARIANT, int ROWS>
__global__ __launch_bounds__(kQuantizeThreads) void QuantizeRowsTiledKernel(
    const float* __restrict__ input, int batches, int depth, size_t tile_bytes,
    int8_t* __restrict__ tiled, float* __restrict__ scaling_factors,
    int32_t* __restrict__ zero_points) {
  using Placement = std::conditional_t<ROWS == kWide, Tile32x32Placement, Tile16x64Placement>;
  // Workgroups are dealt round-robin to the 8 XCDs: the rows of a tile go to one XCD, in whose L2
  // their 16-byte pieces of a line meet (with a tile's rows on eight XCDs every line leaves as
  // eight partial writes: 2048 rows of 4096 13.1 us, now 10.5). Whole rounds of 8 tiles; what is
  // left of the grid keeps its order.
  int m = blockIdx.x;
  if (m < static_cast<int>(gridDim.x / (8 * ROWS) * (8 * ROWS))) {
    const int in_round = m % (8 * ROWS);
    m += (in_round % 8) * ROWS + in_round / 8 - in_round;
  }
  int8_t* tile_row = tiled + static_cast<size_t>(m / ROWS) * tile_bytes;
  const Placement place{m % ROWS};
  if (m < batches) {
    // EvalBlockwise4Bit always quantizes asymmetrically (fully_connected.cc:1044-1047).
    QuantizeRow<VARIANT, Placement>(input + static_cast<size_t>(m) * depth, depth, tile_row, depth,
                                    scaling_factors + m, zero_points + m, /*do_asymmetric=*/1, place);
  } else {
    for (int k = threadIdx.x * 8; k < depth; k += kQuantizeThreads * 8) {
      *reinterpret_cast<uint2*>(tile_row + place(k)) = make_uint2(0, 0);
    }
  }
}

struct GemmArgs {
  const char* filter;       // tile32x32s
  const char* scales;       // float32 [tiles][quads of blocks][32 channels][4 blocks]
  const char* activations;  // tile16x64 or tile32x32
  const float* scaling_factors;  // [batches]
  const int32_t* zero_points;    // [batches]
  const float* kfsum;            // [out_depth]
  const float* bias;             // [out_depth] or nullptr
  float* output;                 // [batches, out_depth]
  int batches, out_depth, nb;
  int channel_tiles, row_tiles;  // of the kernel's tile size
};

// Lane j of every 16 lanes to all 16 (row_newbcast:j).
template <int J>
__device__ __forceinline__ float RowBroadcast(float v) {
  // Every lane has a source lane, so no previous value is kept: the move can then merge into
  // the multiply that uses it.
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + J, 0xF, 0xF, true));
}

// A block sum that an MFMA left on top of the bit pattern of kSumBase is, read as a float,
// kSumBase + sum; see the head of this file.
constexpr float kSumBase = 12582912.0f;  // 1.5 * 2^23
constexpr int kSumBaseBits = 0x4B400000;
// float(sum) * scale, rounded once; `offset` is -kSumBase * scale.
__device__ __forceinline__ float ScaleBlockSum(int biased_sum, float scale, float offset) {
  return __fmaf_rn(__int_as_float(biased_sum), scale, offset);
}

// Under an infinite scale (a model's own) that form gives NaN where the product is infinite. A
// wavefront that ends its walk with a NaN therefore walks its tiles again with conversion and
// product apart: only then, so the loop above pays nothing for it.
template <int N>
__device__ __forceinline__ bool AnyNaN(const float (&v)[N]) {
  bool any = false;
#pragma unroll
  for (int i = 0; i < N; ++i) any = any || v[i] != v[i];
  return any;
}

// fully_connected.cc:1078-1082: zero-point term, row scale, bias.
__device__ __forceinline__ float FinishOutput(float sum, float zero_point, float kfsum,
                                              float row_scale, bool has_bias, float bias) {
  const float v = __fmul_rn(__fsub_rn(sum, __fmul_rn(zero_point, kfsum)), row_scale);
  return has_bias ? __fadd_rn(v, bias) : v;
}

// Workgroups are dealt round-robin to the 8 XCDs: each XCD gets a contiguous range of ids, and ids
// walk rectangles of 8 workgroup rows x all channels, the rows fastest, so that the workgroups
// resident on an XCD share their operands in its L2. The grid is rounded up to whole rounds of 8; false:
// a workgroup of that padding. (Only grids that were such rounds were dealt out like this before:
// 128 x 6144 -> 9000, 284 workgroups, filters not in the cache, 63 -> 54 us; 200 rows 72 -> 52.)
__device__ __forceinline__ bool WorkgroupTile(int wgs_c, int wgs_r, int* wg_c, int* wg_r) {
  const int per_xcd = static_cast<int>(gridDim.x / 8);
  const int id = static_cast<int>(blockIdx.x % 8) * per_xcd + static_cast<int>(blockIdx.x / 8);
  if (id >= wgs_c * wgs_r) return false;
  const int band = id / (8 * wgs_c);
  const int band_rows = min(8, wgs_r - 8 * band);
  const int in_band = id - band * 8 * wgs_c;
  *wg_r = 8 * band + in_band % band_rows;
  *wg_c = in_band / band_rows;
  return true;
}

// RT tiles of 16 channels x 16 rows per wavefront, the four of a workgroup on four channel tiles. PAIRS:
// pairs of blocks in flight.
template <int RT, int PAIRS>
__global__ __launch_bounds__(kThreads, 2) void FcInt4BlockwiseGemmKernel(GemmArgs a, int wgs_c,
                                                                         int wgs_r) {
  const int lane = threadIdx.x & 63;
  // The wavefront index as a scalar: tile addresses then stay in scalar registers and every
  // load is "scalar base + lane offset".
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int wg_c, wg_r;
  if (!WorkgroupTile(wgs_c, wgs_r, &wg_c, &wg_r)) return;
  const int ct = wg_c * 4 + wave;
  const int rt0 = wg_r * RT;
  if (ct >= a.channel_tiles || rt0 >= a.row_tiles) return;
  const int nb = a.nb;
  const int pairs = (nb + 1) / 2, quads = (nb + 3) / 4;
  // Half of a tile of 32 channels, by lane offsets: 8 bytes of each of the pair's blocks.
  const char* const wp = a.filter + static_cast<size_t>(ct >> 1) * nb * 1024 + (ct & 1) * 256;
  const char* const sp = a.scales + static_cast<size_t>(ct >> 1) * quads * 512 + (ct & 1) * 256;
  const char* xp[RT];
  // Row tiles past the edge re-read the last valid one; their outputs are never stored.
#pragma unroll
  for (int j = 0; j < RT; ++j) {
    xp[j] = a.activations + static_cast<size_t>(min(rt0 + j, a.row_tiles - 1)) * pairs * 1024;
  }
  // Operands of pair p in slot p % PAIRS, scales of quad q (four blocks) in slot q % kSlots. A slot
  // is requested again right behind the last operation that reads it, so that the loads land in
  // the registers they are read from. Past the end: a hot line, result unused.
  constexpr int kSlots = PAIRS <= 4 ? 2 : PAIRS / 2;
  i64 w[PAIRS][2];
  i64x2 x[PAIRS][RT];
  float4 sg[kSlots];
  uint32_t lane16 = lane * 16, channel16 = (lane & 15) * 16;
  uint32_t weight8 = channel16 + (lane >> 5) * 512 + ((lane >> 4) & 1) * 8;
  auto fetch = [&](auto slot, int p) {
    constexpr int s = decltype(slot)::value;
    const int pp = min(p, pairs - 1);
    const size_t at = static_cast<size_t>(pp) * 1024;
#pragma unroll
    for (int j = 0; j < RT; ++j) x[s][j] = *reinterpret_cast<const i64x2*>(xp[j] + at + lane16);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // An odd block count: the last pair's second block is the first again, under zero scales.
      const size_t block = static_cast<size_t>(min(2 * pp + h, nb - 1)) * 1024;
      w[s][h] = *reinterpret_cast<const i64*>(wp + block + weight8);
    }
  };
  auto fetch_scales = [&](auto slot, int q) {
    constexpr int s = decltype(slot)::value;
    const size_t at = static_cast<size_t>(min(q, quads - 1)) * 512;
    sg[s] = *reinterpret_cast<const float4*>(sp + at + channel16);
  };
  // One request at a time, in this order: waits count from the newest.
  StaticFor<kSlots>([&](auto q) {
    fetch_scales(q, decltype(q)::value);
    __builtin_amdgcn_sched_barrier(0);
  });
  StaticFor<PAIRS>([&](auto s) {
    fetch(s, decltype(s)::value);
    __builtin_amdgcn_sched_barrier(0);
  });

  // out[rj][i]: channel 16 ct + lane % 16, batch row 16 (rt0 + rj) + 4 (lane / 16) + i.
  float out[RT][4];
#pragma unroll
  for (int rj = 0; rj < RT; ++rj)
#pragma unroll
    for (int i = 0; i < 4; ++i) out[rj][i] = 0.0f;

  i32x4 base_bits = {kSumBaseBits, kSumBaseBits, kSumBaseBits, kSumBaseBits};
  asm volatile("" : "+v"(base_bits));  // in registers for good
  // The vector work on a tile trails its MFMA by kLag tiles, in this order (the fences keep it): the
  // matrix core works on the next tiles meanwhile.
  constexpr int kTiles = RT;  // tiles per block
  constexpr int kLag = 3;
  // The tiles of pairs first .. first + COUNT - 1 (first a multiple of the slot counts; pair u of
  // them in slots u % PAIRS and u / 2 % kSlots).
  auto walk = [&](auto count_c, auto from_c, auto refill_c, int first) {
    constexpr int kCount = decltype(count_c)::value, kFrom = decltype(from_c)::value;
    constexpr bool kRefill = decltype(refill_c)::value;
    constexpr int kAll = kCount * 2 * kTiles;
    // (Opaque here, or the lane's offset is folded into every pointer outside the loop and each
    // load pays a 64-bit vector addition for the pair's instead.)
    asm volatile("" : "+v"(lane16), "+v"(channel16), "+v"(weight8));
    i32x4 acc[kLag + 1];
    StaticFor<kAll + kLag>([&](auto t_const) {
      constexpr int t = decltype(t_const)::value;
      if constexpr (t < kAll) {
        constexpr int u = kFrom + t / (2 * kTiles), at = t % (2 * kTiles);
        constexpr int h = at / kTiles, rj = at % RT;
        constexpr int s = u % PAIRS;
        acc[t % (kLag + 1)] = __builtin_amdgcn_mfma_i32_16x16x32_i8(x[s][rj][h], w[s][h],
                                                                    base_bits, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (kRefill && at == 2 * kTiles - 1) {
          fetch(std::integral_constant<int, s>{}, first + u + PAIRS);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if constexpr (t >= kLag) {
        constexpr int d = t - kLag;
        constexpr int u = kFrom + d / (2 * kTiles), at = d % (2 * kTiles);
        constexpr int h = at / kTiles, rj = at % RT;
        constexpr int b = 2 * (u % 2) + h, cur = u / 2 % kSlots;  // block of which quad
        const float4& q = sg[cur];
        const float scale = b == 0 ? q.x : b == 1 ? q.y : b == 2 ? q.z : q.w;
        const float offset = __fmul_rn(-kSumBase, scale);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          out[rj][i] =
              __fadd_rn(out[rj][i], ScaleBlockSum(acc[d % (kLag + 1)][i], scale, offset));
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (kRefill && u % 2 == 1 && at == 2 * kTiles - 1) {
          fetch_scales(std::integral_constant<int, cur>{}, (first + u) / 2 + kSlots);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    });
  };
  // Whole turns of both rings are straight lines (slots are compile-time constants, and there is no
  // branch to move registers at); what is left of the depth goes pair by pair.
  constexpr int kTrip = PAIRS > 2 * kSlots ? PAIRS : 2 * kSlots;
  static_assert(kTrip % PAIRS == 0 && kTrip % (2 * kSlots) == 0, "trip");
  using std::integral_constant;
  int first = 0;
  for (; first + kTrip <= pairs; first += kTrip) {
    walk(integral_constant<int, kTrip>{}, integral_constant<int, 0>{}, std::true_type{}, first);
  }
  StaticFor<kTrip - 1>([&](auto u_const) {
    constexpr int u = decltype(u_const)::value;
    if (first + u < pairs) {
      walk(integral_constant<int, 1>{}, integral_constant<int, u>{}, std::false_type{}, first);
      // Beyond the slots that a whole turn leaves filled (a ring shorter than the trip).
      if constexpr (u + PAIRS < kTrip - 1) fetch(integral_constant<int, u % PAIRS>{}, first + u + PAIRS);
    }
  });
  bool nan = false;
#pragma unroll
  for (int rj = 0; rj < RT; ++rj) nan = nan || AnyNaN(out[rj]);
  if (__ballot(nan) != 0) {
    const i32x4 zero = {0, 0, 0, 0};
#pragma unroll
    for (int rj = 0; rj < RT; ++rj) {
      float again[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      for (int b = 0; b < nb; ++b) {
        const float scale = *reinterpret_cast<const float*>(sp + static_cast<size_t>(b / 4) * 512 +
                                                            channel16 + (b % 4) * 4);
        const i64 wb = *reinterpret_cast<const i64*>(wp + static_cast<size_t>(b) * 1024 + weight8);
        const i64x2 xb = *reinterpret_cast<const i64x2*>(xp[rj] + static_cast<size_t>(b / 2) * 1024 + lane16);
        const i32x4 acc = __builtin_amdgcn_mfma_i32_16x16x32_i8(b % 2 ? xb[1] : xb[0], wb, zero, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          again[i] = __fadd_rn(again[i], __fmul_rn(static_cast<float>(acc[i]), scale));
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) out[rj][i] = again[i];
    }
  }

#pragma unroll
  for (int rj = 0; rj < RT; ++rj) {
    const int m0 = (rt0 + rj) * kTile + 4 * (lane >> 4);
    float zp[4], row_scale[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = min(m0 + i, a.batches - 1);
      zp[i] = static_cast<float>(a.zero_points[m]);
      row_scale[i] = a.scaling_factors[m];
    }
    const int n = ct * kTile + (lane & 15);
    if (n >= a.out_depth) continue;
    const float kfsum = a.kfsum[n];
    const float bias = a.bias ? a.bias[n] : 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float v = FinishOutput(out[rj][i], zp[i], kfsum, row_scale[i], a.bias != nullptr, bias);
      if (m0 + i < a.batches) a.output[static_cast<size_t>(m0 + i) * a.out_depth + n] = v;
    }
  }
}


// The large form: CT x RT tiles of 32 channels x 32 rows per wavefront, four wavefronts in WROWS x
// 4 / WROWS; BLOCKS blocks in flight. Per tile and block one MFMA (32 cycles of the matrix core) and
// 32 vector operations on its 16 results per lane (72 cycles of the SIMD from two wavefronts on).
template <int CT, int RT, int WROWS, int BLOCKS>
__global__ __launch_bounds__(kThreads, 2) void FcInt4BlockwiseGemmLargeKernel(GemmArgs a, int wgs_c,
                                                                              int wgs_r) {
  using i32x16 = int __attribute__((ext_vector_type(16)));
  constexpr int WCH = 4 / WROWS;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int wg_c, wg_r;
  if (!WorkgroupTile(wgs_c, wgs_r, &wg_c, &wg_r)) return;
  const int ct0 = (wg_c * WCH + wave % WCH) * CT;
  const int rt0 = (wg_r * WROWS + wave / WCH) * RT;
  if (ct0 >= a.channel_tiles || rt0 >= a.row_tiles) return;
  const int nb = a.nb;
  const int quads = (nb + 3) / 4;
  const char* wp[CT];
  const char* sp[CT];
  const char* xp[RT];
#pragma unroll
  for (int j = 0; j < CT; ++j) {
    const int ct = min(ct0 + j, a.channel_tiles - 1);
    wp[j] = a.filter + static_cast<size_t>(ct) * nb * 1024;
    sp[j] = a.scales + static_cast<size_t>(ct) * quads * 512;
  }
#pragma unroll
  for (int j = 0; j < RT; ++j) {
    xp[j] = a.activations + static_cast<size_t>(min(rt0 + j, a.row_tiles - 1)) * nb * 1024;
  }
  // Operands of block b in slot b % BLOCKS, scales of quad q in slot q % 2; requested again behind
  // the last operation that reads them, as above.
  i32x4 w[BLOCKS][CT], x[BLOCKS][RT];
  float4 sg[2][CT];
  uint32_t lane16 = lane * 16, channel16 = (lane & 31) * 16;
  auto fetch = [&](auto slot, int b) {
    constexpr int s = decltype(slot)::value;
    const size_t at = static_cast<size_t>(min(b, nb - 1)) * 1024;
#pragma unroll
    for (int j = 0; j < RT; ++j) x[s][j] = *reinterpret_cast<const i32x4*>(xp[j] + at + lane16);
#pragma unroll
    for (int j = 0; j < CT; ++j) w[s][j] = *reinterpret_cast<const i32x4*>(wp[j] + at + lane16);
  };
  auto fetch_scales = [&](auto slot, int q) {
    constexpr int s = decltype(slot)::value;
    const size_t at = static_cast<size_t>(min(q, quads - 1)) * 512;
#pragma unroll
    for (int j = 0; j < CT; ++j) sg[s][j] = *reinterpret_cast<const float4*>(sp[j] + at + channel16);
  };
  StaticFor<2>([&](auto q) {
    fetch_scales(q, decltype(q)::value);
    __builtin_amdgcn_sched_barrier(0);
  });
  StaticFor<BLOCKS>([&](auto s) {
    fetch(s, decltype(s)::value);
    __builtin_amdgcn_sched_barrier(0);
  });

  // out[cj][rj][e]: channel 32 (ct0 + cj) + lane % 32,
  // batch row 32 (rt0 + rj) + 8 (e / 4) + 4 (lane / 32) + e % 4.
  float out[CT][RT][16];
#pragma unroll
  for (int cj = 0; cj < CT; ++cj)
#pragma unroll
    for (int rj = 0; rj < RT; ++rj)
#pragma unroll
      for (int e = 0; e < 16; ++e) out[cj][rj][e] = 0.0f;

  i32x16 base_bits;
#pragma unroll
  for (int e = 0; e < 16; ++e) base_bits[e] = kSumBaseBits;
  asm volatile("" : "+v"(base_bits));  // in registers for good
  constexpr int kTiles = CT * RT;
  // The tiles of blocks first + kFrom ... (kCount of them), the vector work one tile behind the MFMAs.
  auto walk = [&](auto count_c, auto from_c, auto refill_c, int first) {
    constexpr int kCount = decltype(count_c)::value, kFrom = decltype(from_c)::value;
    constexpr bool kRefill = decltype(refill_c)::value;
    constexpr int kAll = kCount * kTiles;
    asm volatile("" : "+v"(lane16), "+v"(channel16));
    i32x16 acc[2];
    StaticFor<kAll + 1>([&](auto t_const) {
      constexpr int t = decltype(t_const)::value;
      if constexpr (t < kAll) {
        constexpr int u = kFrom + t / kTiles, cj = t % kTiles / RT, rj = t % RT;
        constexpr int s = u % BLOCKS;
        acc[t % 2] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x[s][rj], w[s][cj], base_bits, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (kRefill && t % kTiles == kTiles - 1) {
          fetch(std::integral_constant<int, s>{}, first + u + BLOCKS);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if constexpr (t >= 1) {
        constexpr int d = t - 1;
        constexpr int u = kFrom + d / kTiles, cj = d % kTiles / RT, rj = d % RT;
        constexpr int b = u % 4, cur = u / 4 % 2;
        const float4& q = sg[cur][cj];
        const float scale = b == 0 ? q.x : b == 1 ? q.y : b == 2 ? q.z : q.w;
        const float offset = __fmul_rn(-kSumBase, scale);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          out[cj][rj][e] = __fadd_rn(out[cj][rj][e], ScaleBlockSum(acc[d % 2][e], scale, offset));
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (kRefill && b == 3 && d % kTiles == kTiles - 1) {
          fetch_scales(std::integral_constant<int, cur>{}, (first + u) / 4 + 2);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    });
  };
  constexpr int kTrip = 8;
  static_assert(kTrip % BLOCKS == 0, "trip");
  using std::integral_constant;
  int first = 0;
  for (; first + kTrip <= nb; first += kTrip) {
    walk(integral_constant<int, kTrip>{}, integral_constant<int, 0>{}, std::true_type{}, first);
  }
  StaticFor<kTrip - 1>([&](auto u_const) {
    constexpr int u = decltype(u_const)::value;
    if (first + u < nb) {
      walk(integral_constant<int, 1>{}, integral_constant<int, u>{}, std::false_type{}, first);
      if constexpr (u + BLOCKS < kTrip - 1) {
        fetch(integral_constant<int, u % BLOCKS>{}, first + u + BLOCKS);
      }
    }
  });
  bool nan = false;
#pragma unroll
  for (int cj = 0; cj < CT; ++cj)
#pragma unroll
    for (int rj = 0; rj < RT; ++rj) nan = nan || AnyNaN(out[cj][rj]);
  if (__ballot(nan) != 0) {
    i32x16 zero;
#pragma unroll
    for (int e = 0; e < 16; ++e) zero[e] = 0;
#pragma unroll
    for (int cj = 0; cj < CT; ++cj) {
#pragma unroll
      for (int rj = 0; rj < RT; ++rj) {
        float again[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) again[e] = 0.0f;
        for (int b = 0; b < nb; ++b) {
          const float scale = *reinterpret_cast<const float*>(sp[cj] + static_cast<size_t>(b / 4) * 512 +
                                                              channel16 + (b % 4) * 4);
          const size_t at = static_cast<size_t>(b) * 1024 + lane16;
          const i32x16 acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(
              *reinterpret_cast<const i32x4*>(xp[rj] + at), *reinterpret_cast<const i32x4*>(wp[cj] + at),
              zero, 0, 0, 0);
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            again[e] = __fadd_rn(again[e], __fmul_rn(static_cast<float>(acc[e]), scale));
          }
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) out[cj][rj][e] = again[e];
      }
    }
  }

#pragma unroll
  for (int rj = 0; rj < RT; ++rj) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int m0 = (rt0 + rj) * kWide + 8 * g + 4 * (lane >> 5);
      float zp[4], row_scale[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = min(m0 + i, a.batches - 1);
        zp[i] = static_cast<float>(a.zero_points[m]);
        row_scale[i] = a.scaling_factors[m];
      }
#pragma unroll
      for (int cj = 0; cj < CT; ++cj) {
        const int n = (ct0 + cj) * kWide + (lane & 31);
        if (n >= a.out_depth) continue;
        const float kfsum = a.kfsum[n];
        const float bias = a.bias ? a.bias[n] : 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float v = FinishOutput(out[cj][rj][4 * g + i], zp[i], kfsum, row_scale[i],
                                       a.bias != nullptr, bias);
          if (m0 + i < a.batches) a.output[static_cast<size_t>(m0 + i) * a.out_depth + n] = v;
        }
      }
    }
  }
}


// ---- the same product on a filter that stays 4 bits per weight --------------------------
//
// For batches between decode and prefill (5 to a few dozen rows) the filter stream bounds the
// kernel above, and sign-extending the nibbles to int8 at prepare doubles that stream. Here
// the filter stays packed (`tile16x128n`) and a wavefront expands a block's nibbles itself,
// three vector operations per block and 16 channels: for channel tile t and quad q of blocks
// (128 depth positions), 1 KiB: lane L's 16 bytes are four dwords, dword j for block 4 q + j,
// channel 16 t + L % 16, depths 8 (L / 16) ... + 8 of that block; byte k of a dword holds
// weight k of those eight in its low nibble and weight k + 4 in its high one (two's
// complement, as in the model). `(d << 4) & 0xF0F0F0F0` and `d & 0xF0F0F0F0` are then the
// eight weights as int8 values 16 w, in depth order: the A operand of v_mfma_i32_16x16x32_i8.
// Every block sum comes out multiplied by 16, hence every product and every partial sum of an
// output (scaling by a power of two commutes with each rounding; fp16 scales times integers
// stay far from the float32 range limits), and the finished sum is multiplied by 1/16 once.
// Behind the weight tiles lie the block scales as fp16: per channel tile and group of 16
// blocks, 512 bytes, lane L's 8 bytes = block 16 g + L % 16, channels 4 (L / 16) ... + 4.
// Activations: `tile16x64`, as above. One channel tile per wavefront (these batch sizes want
// the filter stream spread over as many wavefronts as possible).


__global__ __launch_bounds__(kThreads) void PackInt4BlockwiseNibblesKernel(
    const uint8_t* __restrict__ filter, const uint16_t* __restrict__ scales_f16, int out_depth,
    int depth, int tiles, int nb, int nq, int ng, uint8_t* __restrict__ dst) {
  const int64_t slot = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  const int64_t slots = static_cast<int64_t>(tiles) * nq * 64;  // 16-byte lane slots
  if (slot < slots) {
    const int lane = static_cast<int>(slot & 63);
    const int64_t tq = slot >> 6;
    const int q = static_cast<int>(tq % nq);
    const int t = static_cast<int>(tq / nq);
    const int n = t * kTile + (lane & 15);
    uint32_t d[4] = {0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int b = 4 * q + j;
      if (n < out_depth && b < nb) {
        // the slice's 8 weights lie in 4 consecutive bytes of the model's row: byte m holds
        // weights 2 m (low nibble) and 2 m + 1 (high nibble)
        const uint8_t* src = filter + static_cast<size_t>(n) * (depth / 2) + b * (kBlock / 2) +
                             4 * (lane >> 4);
        uint32_t w[8];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          w[2 * m] = src[m] & 0xFu;
          w[2 * m + 1] = src[m] >> 4;
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) d[j] |= (w[k] | (w[k + 4] << 4)) << (8 * k);
      }
    }
    reinterpret_cast<uint4*>(dst)[slot] = make_uint4(d[0], d[1], d[2], d[3]);
  }
  // scales: one thread per (tile, group of 16 blocks, lane)
  const int64_t scale_slots = static_cast<int64_t>(tiles) * ng * 64;
  if (slot < scale_slots) {
    const int lane = static_cast<int>(slot & 63);
    const int64_t tg = slot >> 6;
    const int g = static_cast<int>(tg % ng);
    const int t = static_cast<int>(tg / ng);
    const int b = 16 * g + (lane & 15);
    uint16_t h[4] = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = t * kTile + 4 * (lane >> 4) + i;
      if (n < out_depth && b < nb) h[i] = scales_f16[static_cast<size_t>(n) * nb + b];
    }
    uint2* out = reinterpret_cast<uint2*>(dst + slots * 16);
    out[slot] = make_uint2(h[0] | (static_cast<uint32_t>(h[1]) << 16),
                           h[2] | (static_cast<uint32_t>(h[3]) << 16));
  }
}

struct NibbleGemmArgs {
  const i32x4* filter;      // tile16x128n
  const uint2* scales;      // fp16 [tiles][ng][64 lanes][4]
  const i64x2* activations;  // tile16x64
  const float* scaling_factors;
  const int32_t* zero_points;
  const float* kfsum;
  const float* bias;
  float* output;
  int batches, out_depth, nb;
  int channel_tiles, row_tiles;
  int vector_store;
};

// A wavefront alone on its SIMD issues a vector operation every 8 cycles or so, and a block takes
// 15 of them; with a branch per block, behind which each MFMA waited for the conversions and
// additions of the one before, 14336 x 4096 at 16 rows took 16.9 us with the row quantizer, now
// 13.5 us. One, two and four groups of 16 blocks in flight measure the same. Row tiles are
// wavefronts of their own for the same reason (32 rows 19.0 us, as two tiles of one wavefront 22.3),
// next to each other on one XCD, or the second fetches the filter from memory once more. Filters
// that give every SIMD more than one wavefront by their channels alone (kPairedMinTiles) are bound
// by that vector work itself, of which the expanded nibbles are shared by two tiles of one
// wavefront (32 rows, filters not in the cache, us: one tile each in any order / on one XCD / two
// tiles: 8192 -> 28672 68.5 / 61.5 / 49.6, 4096 -> 32000 39.6 / 34.2 / 29.3).
// The wavefronts of the 4-bit-resident kernels share nothing (no LDS image, no barrier), so each is
// a workgroup of its own: the dispatcher then spreads them one by one over the compute units.
// In workgroups of four, a launch of 2304 wavefronts leaves 64 compute units with three
// workgroups and the rest with two, and takes as long as three everywhere (36864 x 16384 at four
// rows: 84 us; as single wavefronts 71 us; 28672 x 16384: 59.6 -> 54.5 us).
constexpr int kLoneWave = 64;

// RT: row tiles per wavefront; WQ, XQ: quads of blocks whose weights / activations are in flight.
template <int RT, int WQ, int XQ>
__global__ __launch_bounds__(kLoneWave, 2) void FcInt4NibbleGemmKernel(NibbleGemmArgs a) {
  const int lane = threadIdx.x & 63;
  // Workgroups are dealt round-robin to the 8 XCDs: the row tiles of a channel tile follow each other
  // on one XCD, in whose L2 the second finds what the first has fetched.
  const int in_xcd = static_cast<int>(blockIdx.x / 8);
  const int row_groups = (a.row_tiles + RT - 1) / RT;
  const int rt0 = in_xcd % row_groups * RT;
  const int ct0 = in_xcd / row_groups * 8 + static_cast<int>(blockIdx.x % 8);
  if (ct0 >= a.channel_tiles) return;
  const int nb = a.nb;
  const int pairs = (nb + 1) / 2;
  const int nq = (nb + 3) / 4;
  const int ng = (nb + 15) / 16;
  const i32x4* wp = a.filter + static_cast<size_t>(ct0) * nq * 64 + lane;
  const uint2* sp = a.scales + static_cast<size_t>(ct0) * ng * 64 + lane;
  const i64x2* xp[RT];  // a last group may be short: its last tile again, not stored
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    xp[r] = a.activations + static_cast<size_t>(min(rt0 + r, a.row_tiles - 1)) * pairs * 64 + lane;
  }
  // Past the end: a hot line, result unused.
  auto fetch_w = [&](int q) {
    return __builtin_nontemporal_load(wp + static_cast<size_t>(min(q, nq - 1)) * 64);
  };
  struct XStage {
    i64x2 x[RT][2];  // blocks 0-1, blocks 2-3 of the quad
  };
  auto fetch_x = [&](int q) {
    const int qq = min(q, nq - 1);
    XStage st;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      st.x[r][0] = xp[r][static_cast<size_t>(min(2 * qq, pairs - 1)) * 64];
      st.x[r][1] = xp[r][static_cast<size_t>(min(2 * qq + 1, pairs - 1)) * 64];
    }
    return st;
  };
  auto fetch_scales = [&](int g) { return sp[static_cast<size_t>(min(g, ng - 1)) * 64]; };
  constexpr int kGroups = WQ / 4;  // scale groups per trip
  static_assert(WQ % 4 == 0 && WQ % XQ == 0, "trip");
  uint2 sg[kGroups];
  i32x4 wring[WQ];
  XStage xring[XQ];
#pragma unroll
  for (int s = 0; s < WQ; ++s) {
    if (s % 4 == 0) sg[s / 4] = fetch_scales(s / 4);
    wring[s] = fetch_w(s);
    if (s < XQ) xring[s] = fetch_x(s);
  }

  // out[r][i]: channel 16 ct0 + 4 (lane / 16) + i, batch row 16 (rt0 + r) + lane % 16, times 16.
  float out[RT][4];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int i = 0; i < 4; ++i) out[r][i] = 0.0f;
  // Whole groups without a branch: the blocks that pad the last group have scales of zero, and
  // adding the zero product leaves a running sum, which is never -0, as it is. A quad's MFMAs are
  // issued ahead of the conversions, products and additions of the quad before it.
  const i32x4 zero = {0, 0, 0, 0};
  float4 scales = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  i32x4 acc[2][4][RT];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int h = 0; h < 4; ++h)
#pragma unroll
      for (int r = 0; r < RT; ++r) acc[u][h][r] = zero;
  auto add_quad = [&](auto u_const) {  // quad u of its group
    constexpr int u = decltype(u_const)::value;
    StaticFor<4>([&](auto h_const) {
      constexpr int h = decltype(h_const)::value;
      constexpr int j = 4 * u + h;  // this block within its scale group
      const float sc[4] = {RowBroadcast<j>(scales.x), RowBroadcast<j>(scales.y),
                           RowBroadcast<j>(scales.z), RowBroadcast<j>(scales.w)};
#pragma unroll
      for (int r = 0; r < RT; ++r) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          out[r][i] =
              __fadd_rn(out[r][i], __fmul_rn(static_cast<float>(acc[u % 2][h][r][i]), sc[i]));
        }
      }
    });
  };
  for (int g = 0; g < ng; g += kGroups) {
    StaticFor<kGroups>([&](auto g_const) {
      constexpr int gi = decltype(g_const)::value;
      if (gi > 0 && g + gi >= ng) return;
      StaticFor<4>([&](auto u_const) {
        constexpr int u = decltype(u_const)::value;  // quad of the group
        constexpr int slot = 4 * gi + u;
        const int quad = 4 * (g + gi) + u;
        const i32x4 w = wring[slot];
        const XStage st = xring[slot % XQ];
        StaticFor<4>([&](auto h_const) {
          constexpr int h = decltype(h_const)::value;
          const uint32_t d = static_cast<uint32_t>(w[h]);
          const uint32_t lo = (d << 4) & 0xF0F0F0F0u;
          const uint32_t hi = d & 0xF0F0F0F0u;
          const i64 wa = static_cast<i64>(static_cast<uint64_t>(lo) |
                                          (static_cast<uint64_t>(hi) << 32));
#pragma unroll
          for (int r = 0; r < RT; ++r) {
            acc[u % 2][h][r] =
                __builtin_amdgcn_mfma_i32_16x16x32_i8(wa, st.x[r][h >> 1][h & 1], zero, 0, 0, 0);
          }
        });
        wring[slot] = fetch_w(quad + WQ);
        xring[slot % XQ] = fetch_x(quad + XQ);
        __builtin_amdgcn_sched_barrier(0);
        add_quad(std::integral_constant<int, (u + 3) % 4>{});  // of the quad before
        if constexpr (u == 0) {
          const uint2 raw = sg[gi];
          scales = make_float4(HalfBitsToFloatFast(static_cast<uint16_t>(raw.x & 0xFFFF)),
                               HalfBitsToFloatFast(static_cast<uint16_t>(raw.x >> 16)),
                               HalfBitsToFloatFast(static_cast<uint16_t>(raw.y & 0xFFFF)),
                               HalfBitsToFloatFast(static_cast<uint16_t>(raw.y >> 16)));
          sg[gi] = fetch_scales(g + gi + kGroups);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    });
  }
  add_quad(std::integral_constant<int, 3>{});

  // fully_connected.cc:1078-1082: zero-point term, row scale, bias -- after taking the factor
  // 16 back out (exact).
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int m = (rt0 + r) * kTile + (lane & 15);
    if (m >= a.batches) return;
    const float zp = static_cast<float>(a.zero_points[m]);
    const float row_scale = a.scaling_factors[m];
    const int n0 = ct0 * kTile + 4 * (lane >> 4);
    float o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = min(n0 + i, a.out_depth - 1);
      o[i] = FinishOutput(__fmul_rn(out[r][i], 0.0625f), zp, a.kfsum[n], row_scale,
                          a.bias != nullptr, a.bias ? a.bias[n] : 0.0f);
    }
    float* dst = a.output + static_cast<size_t>(m) * a.out_depth + n0;
    if (n0 + 3 < a.out_depth && a.vector_store) {
      *reinterpret_cast<float4*>(dst) = make_float4(o[0], o[1], o[2], o[3]);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (n0 + i < a.out_depth) dst[i] = o[i];
      }
    }
  }
}

// The same product where tiles are few (narrow filters): the depth of a tile dealt to the four
// wavefronts of a workgroup. One wavefront that walks it alone takes 46 ns a block, and only the
// additions, a quarter of that, have to be in block order. So wavefront s takes blocks 16 s ...
// + 16 of every 64, leaves their scaled sums in registers (4 per block), and the running outputs
// go from wavefront to wavefront through LDS, four turns with a barrier each, in which a wavefront
// only adds (16 blocks, 4 chains side by side); the operands of its next 16 blocks are requested
// before the turns. Rows are the MFMA's A operand, so a lane's four sums share one channel and one
// scale. Results are bit-identical to the other forms. With the row quantizer, one wavefront per tile -> here: 16 x 4096 -> 4096
// 12.6 -> 10.5 us, 16 x 16384 -> 2048 33.4 -> 26.8 us (the int8-expanded GEMM 48.8). Rounds of 128
// blocks (eight wavefronts, or 32 blocks each) were no faster, and products made in the slots
// between a wavefront's turns slower (244 registers, loads waited for in each slot: 13.6 us).
constexpr int kChainWaves = 4;
constexpr int kChainBlocks = 16;  // per wavefront and round: one scale group, four quads

__global__ __launch_bounds__(kChainWaves * 64, 2) void FcInt4NibbleChainKernel(NibbleGemmArgs a) {
  constexpr int kScaleStride = kChainBlocks + 8;  // halves: 16-byte lines, spread over the banks
  __shared__ float carry[4][64];
  __shared__ __align__(16) uint16_t scale_lines[kChainWaves][kTile][kScaleStride];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ct0 = blockIdx.x, rt0 = blockIdx.y;
  const int nb = a.nb;
  const int pairs = (nb + 1) / 2, nq = (nb + 3) / 4, ng = (nb + 15) / 16;
  const i32x4* wp = a.filter + static_cast<size_t>(ct0) * nq * 64 + lane;
  const uint2* sp = a.scales + static_cast<size_t>(ct0) * ng * 64 + lane;
  const i64x2* xp = a.activations + static_cast<size_t>(rt0) * pairs * 64 + lane;
  uint2 sg;
  i32x4 w[4];
  i64x2 x[4][2];
  auto request = [&](int group) {  // past the end: clamped addresses, results unused
    sg = sp[static_cast<size_t>(min(group, ng - 1)) * 64];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int q = min(4 * group + u, nq - 1);
      w[u] = __builtin_nontemporal_load(wp + static_cast<size_t>(q) * 64);
      x[u][0] = xp[static_cast<size_t>(min(2 * q, pairs - 1)) * 64];
      x[u][1] = xp[static_cast<size_t>(min(2 * q + 1, pairs - 1)) * 64];
    }
  };
  request(wave);

  // The output this lane finishes: register `wave` of the tile, i.e. row 4 (L / 16) + wave, channel
  // L % 16.
  const int m = rt0 * kTile + 4 * (lane >> 4) + wave;
  const int n = ct0 * kTile + (lane & 15);
  const int mc = min(m, a.batches - 1), nc = min(n, a.out_depth - 1);
  const float zp = static_cast<float>(a.zero_points[mc]);
  const float row_scale = a.scaling_factors[mc];
  const float kfsum = a.kfsum[nc];
  const float bias = a.bias ? a.bias[nc] : 0.0f;

  const i32x4 zero = {0, 0, 0, 0};
  uint16_t* const my_lines = &scale_lines[wave][0][0];
  for (int group0 = 0; group0 < ng; group0 += kChainWaves) {
    const int group = group0 + wave;
    // Scales arrive as (block, four channels) per lane and are wanted as (channel, blocks): through
    // LDS of the wavefront's own, whose operations stay in order.
    uint16_t* to = my_lines + (lane >> 4) * 4 * kScaleStride + (lane & 15);
    to[0] = static_cast<uint16_t>(sg.x);
    to[kScaleStride] = static_cast<uint16_t>(sg.x >> 16);
    to[2 * kScaleStride] = static_cast<uint16_t>(sg.y);
    to[3 * kScaleStride] = static_cast<uint16_t>(sg.y >> 16);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    float product[kChainBlocks][4];
    StaticFor<2>([&](auto e_const) {
      constexpr int e = decltype(e_const)::value;
      const i32x4 raw = *reinterpret_cast<const i32x4*>(my_lines + (lane & 15) * kScaleStride + 8 * e);
      StaticFor<8>([&](auto b_const) {
        constexpr int b = 8 * e + decltype(b_const)::value;
        const uint32_t pair = static_cast<uint32_t>(raw[(b % 8) / 2]);
        const float scale = HalfBitsToFloatFast(static_cast<uint16_t>(b % 2 ? pair >> 16 : pair & 0xFFFF));
        const uint32_t d = static_cast<uint32_t>(w[b / 4][b % 4]);
        const uint32_t lo = (d << 4) & 0xF0F0F0F0u;
        const uint32_t hi = d & 0xF0F0F0F0u;
        const i64 wb = static_cast<i64>(static_cast<uint64_t>(lo) | (static_cast<uint64_t>(hi) << 32));
        const i32x4 acc = __builtin_amdgcn_mfma_i32_16x16x32_i8(x[b / 4][(b % 4) / 2][b % 2], wb, zero, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          product[b][i] = __fmul_rn(static_cast<float>(acc[i]), scale);
        }
      });
    });
    const int valid = min(nb - group * kChainBlocks, kChainBlocks);
    request(group + kChainWaves);
    for (int turn = 0; turn < kChainWaves; ++turn) {
      if (turn == wave && valid > 0) {
        float out[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) out[i] = group == 0 ? 0.0f : carry[i][lane];
        StaticFor<kChainBlocks>([&](auto b_const) {
          constexpr int b = decltype(b_const)::value;
          if (b < valid) {
#pragma unroll
            for (int i = 0; i < 4; ++i) out[i] = __fadd_rn(out[i], product[b][i]);
          }
        });
#pragma unroll
        for (int i = 0; i < 4; ++i) carry[i][lane] = out[i];
      }
      __syncthreads();
    }
  }
  // fully_connected.cc:1078-1082, after taking the factor 16 back out (exact).
  if (m < a.batches && n < a.out_depth) {
    a.output[static_cast<size_t>(m) * a.out_depth + n] = FinishOutput(
        __fmul_rn(carry[wave][lane], 0.0625f), zp, kfsum, row_scale, a.bias != nullptr, bias);
  }
}

// The four-wavefront kernel up to this many tiles (two workgroups per CU); with more the chip is
// busy enough that one wavefront per tile moves less (us, wavefronts: 16 x 2976 -> 5003, 313 tiles,
// 10.9 / 11.1; 32 x 4096 -> 4096, 512 tiles, 12.3 / 13.2; 64 x 4096 -> 4096, 1024 tiles, 17.6 / 14.6).
constexpr int kChainMaxTiles = 512;
// Two row tiles per wavefront from this many channel tiles on.
constexpr int kPairedMinTiles = 1536;


// ---- the same filter for one to four rows: four blocks per matrix-core tile ----------------
//
// With at most four batch rows a 16 x 16 result tile per block is three quarters padding, and
// what bounds the kernel above is the vector work per tile (conversion, scale, add: per block
// whatever the row count). Here the sixteen columns of a result tile are (block j of the quad,
// row r), column 4 j + r: the quad's four MFMAs accumulate into ONE tile, MFMA j with a B operand
// that holds the rows' values of block j in columns 4 j .. 4 j + 3 and zeros elsewhere (a lane
// loads the eight activation bytes of its own column's block once per quad; a select under the
// mask "this lane's column belongs to block j" makes the four operands). One
// conversion and one scale per tile instead of four; the products of blocks 1..3 then reach the
// lanes of block 0 by row shifts and are added there in block order, which is the reference's
// order of float additions, so the results are bit-identical to every other form. Rows are read
// from the standard row quantizer's row-major output; there is no LDS image and no barrier.
struct NibbleQuadArgs {
  const i32x4* filter;   // tile16x128n
  const uint2* scales;   // fp16 [tiles][ng][64 lanes][4]
  const int8_t* rows;    // [batches][depth] int8
  const float* scaling_factors;
  const int32_t* zero_points;
  const float* kfsum;
  const float* bias;
  float* output;
  int batches, depth, out_depth, nb, channel_tiles, vector_store;
};

// The value of the lane N places up in the same row of 16 (row_shl:N); lanes past the row read 0.
template <int N>
__device__ __forceinline__ float FromLaneAbove(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x100 + N, 0xF, 0xF, true));
}

template <int WQ, int XQ>
__device__ __forceinline__ void FcInt4NibbleQuadBody(const NibbleQuadArgs& a, int ct0) {
  const int lane = threadIdx.x & 63;
  const int col = lane & 15;
  const int jl = col >> 2;                     // the block of a quad this lane's column belongs to
  const int r = min(col & 3, a.batches - 1);   // its batch row (clamped: the copy is not stored)
  const int nb = a.nb;
  const int nq = (nb + 3) / 4;
  const int ng = (nb + 15) / 16;
  // Every tensor is in global memory. The grouped kernel reads this struct from a table in
  // memory, and pointers that come from memory carry no address space: accesses through them
  // would go the flat path, whose waits also count LDS traffic (the scale broadcasts) and cannot
  // leave the rings of loads in flight. So the address space is stated here.
  const LRTFC_GLOBAL i32x4* wp =
      (const LRTFC_GLOBAL i32x4*)a.filter + static_cast<size_t>(ct0) * nq * 64 + lane;
  using U32x2 = unsigned __attribute__((ext_vector_type(2)));
  using F32x4 = float __attribute__((ext_vector_type(4)));
  const LRTFC_GLOBAL U32x2* sp =
      (const LRTFC_GLOBAL U32x2*)a.scales + static_cast<size_t>(ct0) * ng * 64 + lane;
  const LRTFC_GLOBAL int8_t* g_rows = (const LRTFC_GLOBAL int8_t*)a.rows;
  // This lane's eight activation bytes of quad q lie at rows + x_first + 128 q (clamped to the
  // row's last block: past the depth the weights are zeros).
  const uint32_t x_lane = static_cast<uint32_t>(r) * a.depth + 8 * (lane >> 4);
  const uint32_t x_first = x_lane + jl * kBlock;
  const uint32_t x_last = x_lane + (nb - 1) * kBlock;
  auto fetch_w = [&](int q) {
    return __builtin_nontemporal_load(wp + static_cast<size_t>(min(q, nq - 1)) * 64);
  };
  // Past the depth: the last block again (its weights there are zeros).
  auto fetch_x = [&](int q) {
    const uint32_t at = min(x_first + static_cast<uint32_t>(min(q, nq - 1)) * (4 * kBlock), x_last);
    return *reinterpret_cast<const LRTFC_GLOBAL i64*>(g_rows + at);
  };
  constexpr int kGroups = WQ / 4 + 1 <= 2 ? 2 : (WQ / 4 + 1 <= 4 ? 4 : 8);
  static_assert((kGroups - 1) * 4 >= WQ, "scale groups must lead the weight ring");
  uint2 sg[kGroups];
  auto fetch_scales = [&](int g) {
    const U32x2 raw = sp[static_cast<size_t>(min(g, ng - 1)) * 64];
    return make_uint2(raw.x, raw.y);
  };
#pragma unroll
  for (int g = 0; g + 1 < kGroups; ++g) sg[g] = fetch_scales(g);
  i32x4 wring[WQ];
  i64 xring[XQ];
#pragma unroll
  for (int s = 0; s < WQ; ++s) wring[s] = fetch_w(s);
#pragma unroll
  for (int s = 0; s < XQ; ++s) xring[s] = fetch_x(s);
  // Where quad t of a group of 16 blocks keeps this lane's scales: the lane of this row of 16
  // whose block is 4 t + jl (byte index for ds_bpermute).
  int from[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) from[t] = 4 * ((lane & 48) + 4 * t + jl);

  // out[i]: channel 16 ct0 + 4 (lane / 16) + i, batch row col (lanes with col < 4), times 16.
  float out[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  const i32x4 zero = {0, 0, 0, 0};
  constexpr int kTrip = WQ > 4 * kGroups ? WQ : 4 * kGroups;
  static_assert(kTrip % WQ == 0 && kTrip % XQ == 0 && kTrip % (4 * kGroups) == 0, "trip");
  float4 cur_scales = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  for (int base = 0; base < nq; base += kTrip) {
    StaticFor<kTrip>([&](auto u_const) {
      constexpr int u = decltype(u_const)::value;
      constexpr int cur = (u / 4) % kGroups;
      if constexpr (u % 4 == 0) {
        const uint2 raw = sg[cur];
        cur_scales = make_float4(HalfBitsToFloatFast(static_cast<uint16_t>(raw.x & 0xFFFF)),
                                 HalfBitsToFloatFast(static_cast<uint16_t>(raw.x >> 16)),
                                 HalfBitsToFloatFast(static_cast<uint16_t>(raw.y & 0xFFFF)),
                                 HalfBitsToFloatFast(static_cast<uint16_t>(raw.y >> 16)));
        sg[(cur + kGroups - 1) % kGroups] = fetch_scales((base + u) / 4 + kGroups - 1);
      }
      const i32x4 w = wring[u % WQ];
      wring[u % WQ] = fetch_w(base + u + WQ);
      const i64 x = xring[u % XQ];
      xring[u % XQ] = fetch_x(base + u + XQ);
      if (base + u < nq) {
        i32x4 acc;
        StaticFor<4>([&](auto h_const) {
          constexpr int h = decltype(h_const)::value;
          const uint32_t d = static_cast<uint32_t>(w[h]);
          const uint32_t lo = (d << 4) & 0xF0F0F0F0u;
          const uint32_t hi = d & 0xF0F0F0F0u;
          const i64 wa = static_cast<i64>(static_cast<uint64_t>(lo) |
                                          (static_cast<uint64_t>(hi) << 32));
          if constexpr (h == 0) {
            acc = __builtin_amdgcn_mfma_i32_16x16x32_i8(wa, jl == h ? x : i64{0}, zero, 0, 0, 0);
          } else {
            acc = __builtin_amdgcn_mfma_i32_16x16x32_i8(wa, jl == h ? x : i64{0}, acc, 0, 0, 0);
          }
        });
        constexpr int t = u % 4;
        const float sc[4] = {
            __int_as_float(__builtin_amdgcn_ds_bpermute(from[t], __float_as_int(cur_scales.x))),
            __int_as_float(__builtin_amdgcn_ds_bpermute(from[t], __float_as_int(cur_scales.y))),
            __int_as_float(__builtin_amdgcn_ds_bpermute(from[t], __float_as_int(cur_scales.z))),
            __int_as_float(__builtin_amdgcn_ds_bpermute(from[t], __float_as_int(cur_scales.w)))};
        // Blocks past the depth have zero weights and zero scales: they add +0.0f, which cannot
        // change a sum that has already taken its first block.
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float p = __fmul_rn(static_cast<float>(acc[i]), sc[i]);
          float o = __fadd_rn(out[i], p);
          o = __fadd_rn(o, FromLaneAbove<4>(p));
          o = __fadd_rn(o, FromLaneAbove<8>(p));
          o = __fadd_rn(o, FromLaneAbove<12>(p));
          out[i] = o;
        }
      }
    });
  }

  // fully_connected.cc:1078-1082, after taking the factor 16 back out (exact).
  const int m = col;
  if (m >= a.batches || m >= 4) return;
  const float zp = static_cast<float>(((const LRTFC_GLOBAL int32_t*)a.zero_points)[m]);
  const float row_scale = ((const LRTFC_GLOBAL float*)a.scaling_factors)[m];
  const LRTFC_GLOBAL float* g_kfsum = (const LRTFC_GLOBAL float*)a.kfsum;
  const LRTFC_GLOBAL float* g_bias = (const LRTFC_GLOBAL float*)a.bias;
  const int n0 = ct0 * kTile + 4 * (lane >> 4);
  float o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int n = min(n0 + i, a.out_depth - 1);
    float v = __fsub_rn(__fmul_rn(out[i], 0.0625f), __fmul_rn(zp, g_kfsum[n]));
    v = __fmul_rn(v, row_scale);
    if (a.bias) v = __fadd_rn(v, g_bias[n]);
    o[i] = v;
  }
  LRTFC_GLOBAL float* dst = (LRTFC_GLOBAL float*)a.output + static_cast<size_t>(m) * a.out_depth + n0;
  if (n0 + 3 < a.out_depth && a.vector_store) {
    *reinterpret_cast<LRTFC_GLOBAL F32x4*>(dst) = F32x4{o[0], o[1], o[2], o[3]};
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (n0 + i < a.out_depth) dst[i] = o[i];
    }
  }
}

template <int WQ, int XQ>
__global__ __launch_bounds__(kLoneWave) void FcInt4NibbleQuadKernel(NibbleQuadArgs a) {
  const int ct0 = blockIdx.x;
  if (ct0 >= a.channel_tiles) return;
  FcInt4NibbleQuadBody<WQ, XQ>(a, ct0);
}


// Several filters of one depth in one launch (independent nodes of a graph, as in the decode
// kernel's grouped form): per node its arguments and the index of its first workgroup, in a
// table in device memory; every node's rows are quantized into its own workspace by one launch.
struct NibbleQuadGroupTable {
  int first_block[LRTFC_INT4_GROUP_MAX + 1];
  int reserved[3];
  NibbleQuadArgs node[LRTFC_INT4_GROUP_MAX];
  const float* input_f32[LRTFC_INT4_GROUP_MAX];
};

template <int WQ, int XQ>
__global__ __launch_bounds__(kLoneWave) void FcInt4NibbleQuadGroupedKernel(
    const NibbleQuadGroupTable* __restrict__ table, int count) {
  // The table counts in blocks of four channel tiles (first_block); a workgroup is one wavefront
  // with one tile. first_block is ascending: this block's node is the number of later nodes whose
  // first block is not beyond it (vector loads and ballots, 64 nodes per turn).
  const int lane = threadIdx.x & 63;
  const int block = static_cast<int>(blockIdx.x >> 2);
  int node = 0;
  for (int base = 0; base + 1 < count; base += 64) {
    const int probe = base + lane + 1;
    const bool not_beyond = probe < count && block >= table->first_block[min(probe, count)];
    node += __popcll(__ballot(not_beyond));
  }
  node = __builtin_amdgcn_readfirstlane(node);
  const NibbleQuadArgs a = table->node[node];
  const int ct0 = (block - table->first_block[node]) * 4 + static_cast<int>(blockIdx.x & 3);
  if (ct0 >= a.channel_tiles) return;
  FcInt4NibbleQuadBody<WQ, XQ>(a, ct0);
}

// Workgroup r quantizes row r % batches of node r / batches into that node's workspace
// (EvalBlockwise4Bit always quantizes asymmetrically, fully_connected.cc:1044-1047).
template <int VARIANT, int THREADS = kQuantizeThreads>
__global__ __launch_bounds__(THREADS) void QuantizeNibbleGroupRowsKernel(
    const NibbleQuadGroupTable* __restrict__ table, int batches) {
  const int node = blockIdx.x / batches;
  const int row = blockIdx.x - node * batches;
  const NibbleQuadArgs& a = table->node[node];
  QuantizeRow<VARIANT, RowMajorPlacement, THREADS>(
                       table->input_f32[node] + static_cast<size_t>(row) * a.depth, a.depth,
                       const_cast<int8_t*>(a.rows) + static_cast<size_t>(row) * a.depth, a.depth,
                       const_cast<float*>(a.scaling_factors) + row,
                       const_cast<int32_t*>(a.zero_points) + row, /*do_asymmetric=*/1);
}

}  // namespace

size_t GemmInt4BlockwiseBytes(int out_depth, int depth) {
  const size_t tiles = (static_cast<size_t>(out_depth) + kWide - 1) / kWide;
  const size_t nb = static_cast<size_t>(depth) / kBlock;
  return tiles * (nb * 1024 + (nb + 3) / 4 * kWide * 4 * sizeof(float));
}

bool FcInt4NibbleGemmFewTiles(int batches, int out_depth) {
  return static_cast<int64_t>((batches + kTile - 1) / kTile) * ((out_depth + kTile - 1) / kTile) <=
         kChainMaxTiles;
}

bool FcInt4BlockwiseGemmSupports(int depth, int blocksize) {
  return blocksize == kBlock && depth > 0 && depth % kBlock == 0;
}

hipError_t LaunchPackInt4BlockwiseGemm(const uint8_t* filter, const uint16_t* scales_f16,
                                       int out_depth, int depth, uint8_t* packed,
                                       hipStream_t stream) {
  if (out_depth == 0 || depth == 0) return hipSuccess;
  const int tiles = (out_depth + kWide - 1) / kWide;
  const int nb = depth / kBlock;
  const int64_t slots = static_cast<int64_t>(tiles) * nb * 128;
  const unsigned grid = static_cast<unsigned>((slots + kThreads - 1) / kThreads);
  hipLaunchKernelGGL(PackInt4BlockwiseGemmKernel, dim3(grid), dim3(kThreads), 0, stream, filter,
                     scales_f16, out_depth, depth, tiles, nb, packed);
  return hipGetLastError();
}

// One tile of 16 rows x the depth padded to whole pairs of blocks, or of 32 rows x the depth.
static size_t RowTileBytes(int depth, int rows) {
  return rows == kWide ? static_cast<size_t>(kWide) * depth
                       : static_cast<size_t>(kTile) * ((static_cast<size_t>(depth) + 2 * kBlock - 1) /
                                                       (2 * kBlock) * (2 * kBlock));
}

size_t TiledRowsBytes(int batches, int depth) {
  const size_t narrow = (static_cast<size_t>(batches) + kTile - 1) / kTile * RowTileBytes(depth, kTile);
  const size_t wide = (static_cast<size_t>(batches) + kWide - 1) / kWide * RowTileBytes(depth, kWide);
  return narrow > wide ? narrow : wide;
}

namespace {
template <int ROWS>
hipError_t LaunchTiledQuantizer(const float* input, int variant, int batches, int depth,
                                void* tiled_rows, float* scaling_factors, int32_t* zero_points,
                                hipStream_t stream) {
  const dim3 grid((batches + ROWS - 1) / ROWS * ROWS), block(kQuantizeThreads);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, block, 0, stream, input, batches, depth,
                       RowTileBytes(depth, ROWS), static_cast<int8_t*>(tiled_rows), scaling_factors,
                       zero_points);
    return hipGetLastError();
  };
  switch (variant) {
    case LRTFC_QUANT_NEON_V8: return launch(QuantizeRowsTiledKernel<LRTFC_QUANT_NEON_V8, ROWS>);
    case LRTFC_QUANT_NEON_LEGACY: return launch(QuantizeRowsTiledKernel<LRTFC_QUANT_NEON_LEGACY, ROWS>);
    default: return launch(QuantizeRowsTiledKernel<LRTFC_QUANT_PORTABLE, ROWS>);
  }
}
}  // namespace

hipError_t LaunchFcInt4BlockwiseGemm(const float* input, int variant, float* scaling_factors,
                                     int32_t* zero_points, const uint8_t* gemm_filter,
                                     const float* kfsum, const float* bias, float* output,
                                     int batches, int depth, int out_depth, void* tiled_rows,
                                     hipStream_t stream) {
  if (batches == 0 || out_depth == 0) return hipSuccess;
  const int nb = depth / kBlock;
  GemmArgs a;
  a.filter = reinterpret_cast<const char*>(gemm_filter);
  a.scales = a.filter + static_cast<size_t>((out_depth + kWide - 1) / kWide) * nb * 1024;
  a.activations = static_cast<const char*>(tiled_rows);
  a.scaling_factors = scaling_factors;
  a.zero_points = zero_points;
  a.kfsum = kfsum;
  a.bias = bias;
  a.output = output;
  a.batches = batches;
  a.out_depth = out_depth;
  a.nb = nb;
  auto launch = [&](auto kernel, auto tile_c, int ct, int rt, int wrows) {
    constexpr int kRows = decltype(tile_c)::value;
    if (hipError_t err = LaunchTiledQuantizer<kRows>(input, variant, batches, depth, tiled_rows,
                                                     scaling_factors, zero_points, stream)) {
      return err;
    }
    a.channel_tiles = (out_depth + kRows - 1) / kRows;
    a.row_tiles = (batches + kRows - 1) / kRows;
    const int wgs_c = (a.channel_tiles + 4 / wrows * ct - 1) / (4 / wrows * ct);
    const int wgs_r = (a.row_tiles + wrows * rt - 1) / (wrows * rt);
    hipLaunchKernelGGL(kernel, dim3((static_cast<unsigned>(wgs_c) * wgs_r + 7) / 8 * 8), dim3(kThreads),
                       0, stream, a, wgs_c, wgs_r);
    return hipGetLastError();
  };
  using Narrow = std::integral_constant<int, kTile>;
  using Wide = std::integral_constant<int, kWide>;
  // Tiles per wavefront, by how many the launch has: a wavefront walks the whole depth, so a launch
  // with few tiles wants them on as many wavefronts as there are SIMDs (1024), and one with many
  // wants large ones, which re-read the least. Measured, us with the row quantizer's launch (S: 16 x
  // 16 tiles, L: 32 x 32; channels x rows per wavefront):
  //   rows x depth -> channels       S 1x1   S 1x2   L 1x1   L 1x2   L 2x2
  //   64 x 4096 -> 4096               14.5    16.0    20.1    30.4    53
  //   128 x 4096 -> 4096              22.8    17.6    20.9    31.4    53
  //   200 x 2944 -> 2944              25.8    21.9    17.9    26.5    43
  //   128 x 4096 -> 14336             57.7    43.5    28.8    33.2    55
  //   512 x 4096 -> 4096              67.2    47.5    31.9    36.4    56
  //   256 x 4096 -> 14336              110    71.4    51.5    44.9    58
  //   512 x 4096 -> 14336              214     135    85.6    85.0    79
  //   2048 x 4096 -> 14336             837     516     325     268    267
  const int64_t narrow_tiles = static_cast<int64_t>((out_depth + kTile - 1) / kTile) *
                               ((batches + kTile - 1) / kTile);
  const int64_t wide_tiles = static_cast<int64_t>((out_depth + kWide - 1) / kWide) *
                             ((batches + kWide - 1) / kWide);
  if (narrow_tiles <= 1024) return launch(FcInt4BlockwiseGemmKernel<1, 8>, Narrow{}, 1, 1, 1);
  if (narrow_tiles <= 2048) return launch(FcInt4BlockwiseGemmKernel<2, 4>, Narrow{}, 1, 2, 1);
  if (wide_tiles <= 2560) return launch(FcInt4BlockwiseGemmLargeKernel<1, 1, 1, 8>, Wide{}, 1, 1, 1);
  if (wide_tiles <= 6144) return launch(FcInt4BlockwiseGemmLargeKernel<1, 2, 1, 4>, Wide{}, 1, 2, 1);
  return launch(FcInt4BlockwiseGemmLargeKernel<2, 2, 2, 2>, Wide{}, 2, 2, 2);
}

size_t GemmInt4BlockwiseNibbleBytes(int out_depth, int depth) {
  const size_t tiles = (static_cast<size_t>(out_depth) + kTile - 1) / kTile;
  const size_t nb = static_cast<size_t>(depth) / kBlock;
  return tiles * ((nb + 3) / 4 * 1024 + (nb + 15) / 16 * 512);
}

hipError_t LaunchPackInt4BlockwiseNibbles(const uint8_t* filter, const uint16_t* scales_f16,
                                          int out_depth, int depth, uint8_t* packed,
                                          hipStream_t stream) {
  if (out_depth == 0 || depth == 0) return hipSuccess;
  const int tiles = (out_depth + kTile - 1) / kTile;
  const int nb = depth / kBlock;
  const int nq = (nb + 3) / 4, ng = (nb + 15) / 16;
  const int64_t slots = static_cast<int64_t>(tiles) * nq * 64;
  const unsigned grid = static_cast<unsigned>((slots + kThreads - 1) / kThreads);
  hipLaunchKernelGGL(PackInt4BlockwiseNibblesKernel, dim3(grid), dim3(kThreads), 0, stream,
                     filter, scales_f16, out_depth, depth, tiles, nb, nq, ng, packed);
  return hipGetLastError();
}

hipError_t LaunchFcInt4BlockwiseNibbleGemm(const float* input, int variant,
                                           float* scaling_factors, int32_t* zero_points,
                                           const uint8_t* nibble_filter, const float* kfsum,
                                           const float* bias, float* output, int batches,
                                           int depth, int out_depth, void* tiled_rows,
                                           hipStream_t stream) {
  if (batches == 0 || out_depth == 0) return hipSuccess;
  const int nb = depth / kBlock;
  const int row_tiles = (batches + kTile - 1) / kTile;
  const int channel_tiles = (out_depth + kTile - 1) / kTile;
  if (batches <= 4) {
    // Row-major quantized rows (they fit where the tiled rows of a 16-row tile would lie).
    if (hipError_t err = LaunchBatchQuantize(input, batches, depth, depth, static_cast<int8_t*>(tiled_rows),
                                             scaling_factors, zero_points, /*do_asymmetric=*/1,
                                             variant, stream)) {
      return err;
    }
    NibbleQuadArgs q;
    q.filter = reinterpret_cast<const i32x4*>(nibble_filter);
    q.scales = reinterpret_cast<const uint2*>(
        nibble_filter + static_cast<size_t>(channel_tiles) * ((nb + 3) / 4) * 1024);
    q.rows = static_cast<const int8_t*>(tiled_rows);
    q.scaling_factors = scaling_factors;
    q.zero_points = zero_points;
    q.kfsum = kfsum;
    q.bias = bias;
    q.output = output;
    q.batches = batches;
    q.depth = depth;
    q.out_depth = out_depth;
    q.nb = nb;
    q.channel_tiles = channel_tiles;
    q.vector_store = (out_depth % 4 == 0) && (reinterpret_cast<uintptr_t>(output) % 16 == 0);
    hipLaunchKernelGGL((FcInt4NibbleQuadKernel<8, 4>), dim3(channel_tiles), dim3(kLoneWave), 0,
                       stream, q);
    return hipGetLastError();
  }
  if (hipError_t err = LaunchTiledQuantizer<kTile>(input, variant, batches, depth, tiled_rows,
                                                   scaling_factors, zero_points, stream)) {
    return err;
  }
  NibbleGemmArgs a;
  a.filter = reinterpret_cast<const i32x4*>(nibble_filter);
  a.scales = reinterpret_cast<const uint2*>(
      nibble_filter + static_cast<size_t>(channel_tiles) * ((nb + 3) / 4) * 1024);
  a.activations = static_cast<const i64x2*>(tiled_rows);
  a.scaling_factors = scaling_factors;
  a.zero_points = zero_points;
  a.kfsum = kfsum;
  a.bias = bias;
  a.output = output;
  a.batches = batches;
  a.out_depth = out_depth;
  a.nb = nb;
  a.channel_tiles = channel_tiles;
  a.row_tiles = row_tiles;
  a.vector_store = (out_depth % 4 == 0) && (reinterpret_cast<uintptr_t>(output) % 16 == 0);
  const dim3 grid(channel_tiles, row_tiles);
  if (grid.y > 65535) return hipErrorInvalidValue;
  if (FcInt4NibbleGemmFewTiles(batches, out_depth)) {
    hipLaunchKernelGGL(FcInt4NibbleChainKernel, grid, dim3(kChainWaves * 64), 0, stream, a);
  } else {
    const unsigned columns = (channel_tiles + 7) / 8 * 8;
    if (row_tiles > 1 && channel_tiles >= kPairedMinTiles) {
      hipLaunchKernelGGL((FcInt4NibbleGemmKernel<2, 4, 4>), dim3(columns * ((row_tiles + 1) / 2)),
                         dim3(kLoneWave), 0, stream, a);
    } else {
      hipLaunchKernelGGL((FcInt4NibbleGemmKernel<1, 8, 8>), dim3(columns * row_tiles),
                         dim3(kLoneWave), 0, stream, a);
    }
  }
  return hipGetLastError();
}


size_t Int4NibbleGroupTableBytes() { return sizeof(NibbleQuadGroupTable); }

// With fewer than about one wavefront per SIMD the decode kernel, which splits a channel
// group's depth among wavefronts, is the faster one.
constexpr int kNibbleGroupMinTiles = 1024;

// The grouped launch takes the 4-bit-resident form where it is the faster one: three or four
// rows of filters deeper than 8192, whose rows the decode kernel parks in 64 KB of LDS per
// workgroup (28672 x 16384 at four rows: 64 us here against 82 us there).
bool Int4NibbleGroupWins(int batches, int depth, int total_channel_tiles) {
  return (batches == 3 || batches == 4) && depth > 8192 && depth % kBlock == 0 &&
         total_channel_tiles >= kNibbleGroupMinTiles;
}

hipError_t PrepareInt4NibbleGroup(const lrtfc_int4_group_node* nodes, int count, int batches,
                                  int depth, void* device_table, lrtfc_int4_group_launch* launch,
                                  hipStream_t stream) {
  if (count < 1 || count > LRTFC_INT4_GROUP_MAX || batches < 1 || batches > 4 ||
      depth % kBlock != 0) {
    return hipErrorInvalidValue;
  }
  static NibbleQuadGroupTable host;  // 20 KB: not on the stack
  static std::mutex host_mutex;
  std::lock_guard<std::mutex> lock(host_mutex);
  host = NibbleQuadGroupTable{};
  const int nb = depth / kBlock;
  int next = 0;
  for (int i = 0; i < count; ++i) {
    if (!nodes[i].nibble_filter || !nodes[i].workspace) return hipErrorInvalidValue;
    host.first_block[i] = next;
    NibbleQuadArgs& q = host.node[i];
    const int channel_tiles = (nodes[i].out_depth + kTile - 1) / kTile;
    const ActivationWorkspace w = SplitActivationWorkspace(nodes[i].workspace, batches, depth);
    q.filter = reinterpret_cast<const i32x4*>(nodes[i].nibble_filter);
    q.scales = reinterpret_cast<const uint2*>(
        nodes[i].nibble_filter + static_cast<size_t>(channel_tiles) * ((nb + 3) / 4) * 1024);
    q.rows = w.q;
    q.scaling_factors = w.sf;
    q.zero_points = w.zp;
    q.kfsum = nodes[i].kfsum;
    q.bias = nodes[i].bias;
    q.output = nodes[i].output;
    q.batches = batches;
    q.depth = depth;
    q.out_depth = nodes[i].out_depth;
    q.nb = nb;
    q.channel_tiles = channel_tiles;
    q.vector_store = (nodes[i].out_depth % 4 == 0) &&
                     (reinterpret_cast<uintptr_t>(nodes[i].output) % 16 == 0);
    host.input_f32[i] = nodes[i].input;
    next += (channel_tiles + 3) / 4;
  }
  host.first_block[count] = next;
  hipError_t err = hipMemcpyAsync(device_table, &host, sizeof(host), hipMemcpyHostToDevice, stream);
  if (err == hipSuccess) err = hipStreamSynchronize(stream);  // `host` is reused by the next call
  if (err != hipSuccess) return err;
  launch->count = count;
  launch->grid_blocks = next;
  launch->ksplit = 1;
  launch->groups_per_wave = 1;
  launch->batches = batches;
  launch->depth = depth;
  launch->split_quantize = 1;
  launch->form = LRTFC_INT4_FORM_GEMM_NIBBLES;
  return hipSuccess;
}

hipError_t LaunchFcInt4NibbleGrouped(const void* table, const lrtfc_int4_group_launch& l,
                                     int variant, hipStream_t stream) {
  if (l.count < 1 || l.grid_blocks < 1) return hipSuccess;
  const auto* t = static_cast<const NibbleQuadGroupTable*>(table);
  // This form serves groups deeper than 8192 only: the wide row quantizer.
  const dim3 qgrid(static_cast<unsigned>(l.count) * l.batches), qblock(kQuantizeDeepThreads);
  switch (variant) {
    case LRTFC_QUANT_NEON_V8:
      hipLaunchKernelGGL((QuantizeNibbleGroupRowsKernel<LRTFC_QUANT_NEON_V8, kQuantizeDeepThreads>),
                         qgrid, qblock, 0, stream, t, l.batches);
      break;
    case LRTFC_QUANT_NEON_LEGACY:
      hipLaunchKernelGGL(
          (QuantizeNibbleGroupRowsKernel<LRTFC_QUANT_NEON_LEGACY, kQuantizeDeepThreads>), qgrid,
          qblock, 0, stream, t, l.batches);
      break;
    default:
      hipLaunchKernelGGL((QuantizeNibbleGroupRowsKernel<LRTFC_QUANT_PORTABLE, kQuantizeDeepThreads>),
                         qgrid, qblock, 0, stream, t, l.batches);
      break;
  }
  if (hipError_t err = hipGetLastError()) return err;
  // At most one wavefront per SIMD (narrow, deep filters): each keeps twice the loads in flight
  // (config 5's 18 down projections at four rows, 2304 wavefronts: 82.7 us on the small rings,
  // 90.0 us on the large ones).
  if (l.grid_blocks * 4 <= 1024) {
    hipLaunchKernelGGL((FcInt4NibbleQuadGroupedKernel<16, 8>), dim3(l.grid_blocks * 4),
                       dim3(kLoneWave), 0, stream, t, l.count);
  } else {
    hipLaunchKernelGGL((FcInt4NibbleQuadGroupedKernel<8, 4>), dim3(l.grid_blocks * 4),
                       dim3(kLoneWave), 0, stream, t, l.count);
  }
  return hipGetLastError();
}

}  // namespace lrtfc
