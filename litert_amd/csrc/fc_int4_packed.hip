// Blockwise-int4 FULLY_CONNECTED (EvalBlockwise4Bit, tflite/kernels/fully_connected.cc
// :1014-1086) on a re-tiled filter, block size 32: the streaming form used for decode.
//
// HBM layout ("tile8x64b", built once per constant filter by PackInt4BlockwiseKernel):
// the filter is cut into tiles of 8 output channels x 64 quantization blocks (2048
// depth). A tile is nine consecutive 1 KiB planes: plane j < 8 holds, for lane L, the 16
// bytes (32 nibbles) of channel j, block L; plane 8 holds, for lane L, the eight fp16
// scales of block L for the tile's channels. Nibbles are stored as (w + 8), i.e. XOR 8,
// so that they are small positive bytes for dot4; tiles of one channel group are
// consecutive along the depth. Every load instruction of a wavefront therefore reads
// 1 KiB of consecutive bytes, weights and scales alike, and one lane finishes a block's
// int32 sum alone (8 dot4): sum(w * q) = dot4(w + 8, q) - 8 * sum(q).
//
// A wavefront owns 8 channels over the whole depth. All loads of its first two tiles go
// out first (a ring that is refilled tile by tile for deeper filters); the activation
// rows are quantized (BatchQuantizeFloats, always asymmetric on this path) and staged in
// LDS, split into planes of high and low nibbles that line up with the filter's dwords,
// while the ring fills. The reference then adds float(block_sum) * scale over the blocks
// of a row in block order in float32; that order is kept: the products of a tile are
// parked in LDS and 8 x batch lanes walk them in order, tile after tile, each walk
// overlapping the wait for the next tile's bytes.
#include <type_traits>

#include "kernels.h"
#include "quantize_device.h"

namespace lrtfc {
namespace {

#define LRTFC_GLOBAL __attribute__((address_space(1)))
using f32x4 = float __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWaveSize;
constexpr int kWideThreads = 512;  // single nodes of deep rows
constexpr int kBlock = 32;       // weights per quantization block
constexpr int kTileRows = 8;
constexpr int kTileBlocks = 64;
constexpr int kPlanes = kTileRows + 1;
constexpr int kTileBytes = kPlanes * 1024;
constexpr int kTileVecs = kPlanes * 64;  // i32x4 per tile
constexpr int kRingTiles = 2;
constexpr int kPStride = kTileBlocks + 4;  // floats per (row, batch) line of parked products
constexpr int kMaxGroupNodes = LRTFC_INT4_GROUP_MAX;
constexpr int kMaxGroupsPerWave = 8;  // 64 channels: one lane each when their kfsum is staged
constexpr int kSplitShallowMinBlocks = 1024;  // grouped launches: see PrepareInt4Group
constexpr int kRowPairsSideBySide = 2;        // lrtfc_int4_group_launch.split_quantize
constexpr int kSideBySideMaxBlocks = 256;
constexpr int kPairRound = 256;  // workgroups of a round: one per CU
constexpr int64_t kSideBySideMaxFilterBytes = 24 << 20;

__global__ __launch_bounds__(kThreads) void PackInt4BlockwiseKernel(
    const uint8_t* __restrict__ filter, const uint16_t* __restrict__ scales, int out_depth,
    int depth, int chunks, int64_t total_vecs, uint8_t* __restrict__ dst) {
  const int64_t v = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (v >= total_vecs) return;
  const int lane = static_cast<int>(v & 63);
  const int64_t plane_index = v >> 6;
  const int plane = static_cast<int>(plane_index % kPlanes);
  const int64_t tile = plane_index / kPlanes;
  const int chunk = static_cast<int>(tile % chunks);
  const int group = static_cast<int>(tile / chunks);
  const int nblk = depth / kBlock;
  const int blk = chunk * kTileBlocks + lane;
  const size_t row_bytes = static_cast<size_t>(depth) / 2;
  uint8_t out[16];
  if (plane < kTileRows) {
    const int row = group * kTileRows + plane;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      uint8_t byte = 0;  // weight 0, weight 0
      if (row < out_depth && blk < nblk) byte = filter[row * row_bytes + blk * 16 + t];
      out[t] = byte ^ 0x88;
    }
  } else {
#pragma unroll
    for (int j = 0; j < kTileRows; ++j) {
      const int row = group * kTileRows + j;
      uint16_t s = 0;
      if (row < out_depth && blk < nblk) s = scales[static_cast<size_t>(row) * nblk + blk];
      out[2 * j] = static_cast<uint8_t>(s & 0xFF);
      out[2 * j + 1] = static_cast<uint8_t>(s >> 8);
    }
  }
  *reinterpret_cast<i32x4*>(dst + v * 16) = *reinterpret_cast<const i32x4*>(out);
}

struct Int4PackedArgs {
  const uint8_t* packed;       // tile8x64b
  const float* input_f32;      // fused form
  const int8_t* input_q;       // unfused form: quantized rows + their scales / zero points
  const float* scaling_factors;
  const int32_t* zero_points;
  const float* kfsum;
  const float* bias;
  float* output;
  int batches, depth, out_depth, chunks;
};

// What a wavefront needs before its first loads are on their way: kernels hand it over in preloaded
// registers or from one read of a table's head, and everything else of Int4PackedArgs is read from
// memory behind those loads.
struct Int4Start {
  const uint8_t* packed;
  const void* rows;  // float32 (fused) or int8
  int depth, out_depth, chunks;
};

// Nibble planes of eight consecutive int8 activations (lo = q0..q3, hi = q4..q7 as packed
// bytes): `high` holds (q >> 4) & 15 and `low` holds q & 15 of element i in bits 4i .. 4i + 3,
// the order in which a dword of the filter holds its eight weights. With q = 16 * qh + ql
// (qh signed, ql unsigned) a block's sum(w * q) is 16 * sdot8(w, qh) + udot8(w + 8, ql) -
// 8 * sum(ql): eight 8-way dot products per 32 weights and no nibble unpacking at all.
__device__ __forceinline__ uint32_t CompressNibbles(uint32_t t) {  // bytes 0x0n -> 16 bits
  t = (t | (t >> 4)) & 0x00FF00FFu;
  return (t | (t >> 8)) & 0xFFFFu;
}
__device__ __forceinline__ void NibblePlanes(uint32_t lo, uint32_t hi, int32_t* high,
                                             int32_t* low) {
  *low = static_cast<int32_t>(CompressNibbles(lo & 0x0F0F0F0Fu) |
                              (CompressNibbles(hi & 0x0F0F0F0Fu) << 16));
  *high = static_cast<int32_t>(CompressNibbles((lo >> 4) & 0x0F0F0F0Fu) |
                               (CompressNibbles((hi >> 4) & 0x0F0F0F0Fu) << 16));
}
__device__ __forceinline__ int32_t SDot8(int32_t a, int32_t b, int32_t acc) {
  return __builtin_amdgcn_sdot8(a, b, acc, false);
}
__device__ __forceinline__ uint32_t UDot8(uint32_t a, uint32_t b, uint32_t acc) {
  return __builtin_amdgcn_udot8(a, b, acc, false);
}

// LDS map: [BT][padded depth] activations as nibble planes (per block of 32: four dwords of
// high nibbles, then four of low nibbles); per wavefront [8 * BT][kPStride]
// parked products; the wavefronts' ranges of the rows.
template <int BT, int THREADS = kThreads>
struct Int4Shared {
  int32_t* q;   // dwords: per row padded_depth / 4
  float* p;     // [waves][8 * BT][kPStride]
  float* mm;    // [BT][waves][2]
  float* kb;    // [waves][2][64]: kfsum and bias of the channels a wavefront covers
  float* ob;    // [waves][64 * BT]: finished outputs of those channels
  // Floats of parked products: one tile per wavefront when a wavefront owns a channel group alone; every
  // tile of the group when `ksplit` wavefronts share it (the ordered walk then needs them all). ksplit is
  // a power of two everywhere: a division by it cost every wavefront some 30 scalar and vector
  // instructions ahead of its first load.
  __host__ __device__ static size_t ProductFloats(int chunks, int ksplit) {
    constexpr int waves = THREADS / kWaveSize;
    const size_t tile = static_cast<size_t>(8) * BT * kPStride;
    return ksplit == 1 ? waves * tile
                       : (waves >> __builtin_ctz(ksplit)) * static_cast<size_t>(chunks) * tile;
  }
  __device__ Int4Shared(int8_t* base, int padded, int chunks, int ksplit) {
    constexpr int waves = THREADS / kWaveSize;
    q = reinterpret_cast<int32_t*>(base);
    size_t off = static_cast<size_t>(BT) * padded;
    p = reinterpret_cast<float*>(base + off);
    off += ProductFloats(chunks, ksplit) * 4;
    mm = reinterpret_cast<float*>(base + off);
    kb = mm + BT * waves * 2;
    ob = kb + waves * 2 * 64;
  }
  static size_t Bytes(int padded, int ksplit) {
    constexpr int waves = THREADS / kWaveSize;
    const int chunks = padded / (kTileBlocks * kBlock);
    return static_cast<size_t>(BT) * padded + ProductFloats(chunks, ksplit) * 4 +
           BT * waves * 2 * 4 + waves * 2 * 64 * 4 + waves * 64 * BT * 4;
  }
};

// A chain lane's additions of parked products, in block order; `line` is its line of the first tile, the
// next tile's lies kTileFloats on. Whole tiles: half a tile is read ahead of the additions, the reads of a
// tile take a third as long as its 64 dependent additions.
template <int kTileFloats>
__device__ __forceinline__ float AddWholeTiles(const float* line, int tiles, float out) {
  constexpr int kAhead = kTileBlocks / 8;  // float4 per half tile
  auto read_half = [&](int half, float4* v) {
    const float4* from = reinterpret_cast<const float4*>(
        line + static_cast<size_t>(half >> 1) * kTileFloats + (half & 1) * (kTileBlocks / 2));
#pragma unroll
    for (int j = 0; j < kAhead; ++j) v[j] = from[j];
  };
  auto add_half = [&](const float4* v) {
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      out = __fadd_rn(out, v[j].x);
      out = __fadd_rn(out, v[j].y);
      out = __fadd_rn(out, v[j].z);
      out = __fadd_rn(out, v[j].w);
    }
  };
  float4 even[kAhead], odd[kAhead];
  read_half(0, even);
  for (int half = 0; half < 2 * tiles; half += 2) {
    read_half(half + 1, odd);
    add_half(even);
    read_half(min(half + 2, 2 * tiles - 1), even);
    add_half(odd);
  }
  return out;
}
// A row's last, partial tile: a quarter of a tile at a time, the next one read ahead. Block by block it cost
// a trip to LDS each (filters not in the caches, one row: 1536 -> 1536 5.1 -> 3.8 us, 4608 -> 4096 8.1 ->
// 7.7; four rows of 1152 -> 6912 6.9 -> 6.0; with a test before every four additions 3.9, 7.7, 6.0). The
// products past the last block are +0 (the padding's scales and activations are zero), and a sum that
// starts at +0 is never -0, so they leave it as it is.
__device__ __forceinline__ float AddPartialTile(const float* line, int count, float out) {
  constexpr int kQuarter = kTileBlocks / 4;
  const int quarters = (count + kQuarter - 1) / kQuarter;
  float4 now[kQuarter / 4], next[kQuarter / 4];
#pragma unroll
  for (int j = 0; j < kQuarter / 4; ++j) now[j] = reinterpret_cast<const float4*>(line)[j];
  for (int quarter = 0; quarter < quarters; ++quarter) {
    const float4* from = reinterpret_cast<const float4*>(line + min(quarter + 1, quarters - 1) * kQuarter);
#pragma unroll
    for (int j = 0; j < kQuarter / 4; ++j) next[j] = from[j];
#pragma unroll
    for (int j = 0; j < kQuarter / 4; ++j) {
      out = __fadd_rn(out, now[j].x);
      out = __fadd_rn(out, now[j].y);
      out = __fadd_rn(out, now[j].z);
      out = __fadd_rn(out, now[j].w);
    }
#pragma unroll
    for (int j = 0; j < kQuarter / 4; ++j) now[j] = next[j];
  }
  return out;
}

// GPT: groups of 8 depth positions each thread keeps in registers between the two passes of
// the prologue; the register form covers depth <= GPT * THREADS * 8.
// The work of one workgroup; `block` is its index among the workgroups of this filter.
// gpw: consecutive channel groups one wavefront works through (ksplit == 1 only). Their
// tiles are one contiguous stretch of the filter, so the ring of loads runs on across group
// boundaries and the prologue (the row quantizer) is paid once for all of them.
// ALL > 0: a wavefront has at most ALL tiles (ksplit == 1 and gpw * chunks <= ALL, or one tile of each
// of ksplit == chunks wavefronts, WideDeep) and requests every one of them before it does anything
// else: no refills, one memory round trip per wavefront, and straight-line code whose waits for
// each tile are exact.
template <int N, class F>
__device__ __forceinline__ void StaticFor(F&& f) {
  if constexpr (N > 0) {
    StaticFor<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

// PRE of them go out ahead of the prologue, the rest behind it: a compute unit accepts only
// some tens of KiB of outstanding loads, and a wavefront whose load issue blocks cannot do its
// share of the row quantizer (14336 x 4096, one row: two tiles per wavefront, one ahead, 8.3 us;
// both ahead 9.0 us; four tiles per wavefront all ahead 9.9 us; the refilled ring of two 8.5 us).
template <int BT, bool FUSED, int VARIANT, int GPT, int ALL = 0, int PRE = 0, int THREADS = kThreads>
__device__ __forceinline__ void FcInt4PackedBody(const Int4Start& start, const Int4PackedArgs& a,
                                                 int block, int batch0, int bt, int ksplit, int gpw,
                                                 int8_t* smem) {
  constexpr int kThreads = THREADS, kWaves = THREADS / kWaveSize;

  // Every tensor is in global memory. Pointers that a kernel read from a table in memory
  // carry no address space, and accesses through them would go the flat path, whose waits
  // cannot leave a ring of loads in flight; so the address space is stated here.
  const LRTFC_GLOBAL i32x4* g_packed = (const LRTFC_GLOBAL i32x4*)start.packed;
  const LRTFC_GLOBAL float* g_input_f32 = (const LRTFC_GLOBAL float*)start.rows;
  const LRTFC_GLOBAL int8_t* g_input_q = (const LRTFC_GLOBAL int8_t*)start.rows;
  const LRTFC_GLOBAL float* g_scaling_factors = (const LRTFC_GLOBAL float*)a.scaling_factors;
  const LRTFC_GLOBAL int32_t* g_zero_points = (const LRTFC_GLOBAL int32_t*)a.zero_points;
  const int tid = threadIdx.x;
  const int lane = tid & (kWaveSize - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWaveSize);
  const int depth = start.depth;
  const int chunks = start.chunks;
  const int padded = chunks * kTileBlocks * kBlock;  // depth padded to whole tiles
  const int groups = (start.out_depth + kTileRows - 1) / kTileRows;
  // ksplit wavefronts share one channel group and take its tiles round-robin (deep, narrow
  // filters would otherwise leave most of the chip without a wavefront).
  const int split_bits = __builtin_ctz(ksplit);
  const int kpart = wave & (ksplit - 1);
  const int group_in_wg = wave >> split_bits;
  const int group0 = (block * (kWaves >> split_bits) + group_in_wg) * gpw;  // may run past the last
  const int my_groups = max(0, min(gpw, groups - group0));
  const int ntiles = my_groups * chunks;  // tiles of this wavefront and its depth partners
  const int first_group = min(group0, groups - 1);
  const LRTFC_GLOBAL i32x4* tbase = g_packed +
                       static_cast<size_t>(first_group) * chunks * kTileVecs + lane;
  Int4Shared<BT, THREADS> sh(smem, padded, chunks, ksplit);
  // Activation loads first (raw, branch-free): whatever the prologue waits for must be
  // requested before the weight ring, because vector memory returns in issue order.
  // Each thread owns groups of 8 consecutive depth positions: g = tid + 256 * j.
  constexpr int kGroupsPerThread = GPT;
  float4 xr[BT][kGroupsPerThread][2];
  i32x2 qr[BT][kGroupsPerThread];
  const int groups8 = depth / 8;
  bool in_regs;
  if (FUSED) {
    in_regs = ((reinterpret_cast<uintptr_t>(start.rows) & 15) == 0) &&
              groups8 <= kGroupsPerThread * kThreads;
    if (in_regs) {
#pragma unroll
      for (int b = 0; b < BT; ++b) {
        const LRTFC_GLOBAL float* x = g_input_f32 + static_cast<size_t>(batch0 + min(b, bt - 1)) * depth;
#pragma unroll
        for (int j = 0; j < kGroupsPerThread; ++j) {
          const int g = min(j * kThreads + tid, groups8 - 1);
          const f32x4 lo = *reinterpret_cast<const LRTFC_GLOBAL f32x4*>(x + g * 8);
          const f32x4 hi = *reinterpret_cast<const LRTFC_GLOBAL f32x4*>(x + g * 8 + 4);
          xr[b][j][0] = make_float4(lo.x, lo.y, lo.z, lo.w);
          xr[b][j][1] = make_float4(hi.x, hi.y, hi.z, hi.w);
        }
      }
    } else {
      for (int b = 0; b < bt; ++b) {  // slow form: min/max from memory before the ring
        const LRTFC_GLOBAL float* x = g_input_f32 + static_cast<size_t>(batch0 + b) * depth;
        float mn = 0.0f, mx = 0.0f;
        for (int i = tid; i < depth; i += kThreads) {
          mn = fminf(mn, x[i]);
          mx = fmaxf(mx, x[i]);
        }
        mn = WaveMinF32(mn);
        mx = WaveMaxF32(mx);
        if (lane == 0) {
          sh.mm[(b * kWaves + wave) * 2] = mn;
          sh.mm[(b * kWaves + wave) * 2 + 1] = mx;
        }
      }
    }
  } else {
    in_regs = ((reinterpret_cast<uintptr_t>(start.rows) & 7) == 0) &&
              groups8 <= kGroupsPerThread * kThreads;
    if (in_regs) {
#pragma unroll
      for (int b = 0; b < BT; ++b) {
        const LRTFC_GLOBAL int8_t* x = g_input_q + static_cast<size_t>(batch0 + min(b, bt - 1)) * depth;
#pragma unroll
        for (int j = 0; j < kGroupsPerThread; ++j) {
          const int g = min(j * kThreads + tid, groups8 - 1);
          qr[b][j] = *reinterpret_cast<const LRTFC_GLOBAL i32x2*>(x + g * 8);
        }
      }
    } else {
      for (int b = 0; b < bt; ++b) {
        const LRTFC_GLOBAL int8_t* x = g_input_q + static_cast<size_t>(batch0 + b) * depth;
        for (int g = tid; g < padded / 8; g += kThreads) {
          uint32_t lo = 0, hi = 0;
          if (g < groups8) {
            for (int t = 0; t < 4; ++t) {
              lo |= static_cast<uint32_t>(static_cast<uint8_t>(x[g * 8 + t])) << (8 * t);
              hi |= static_cast<uint32_t>(static_cast<uint8_t>(x[g * 8 + 4 + t])) << (8 * t);
            }
          }
          int32_t high, low;
          NibblePlanes(lo, hi, &high, &low);
          sh.q[b * (padded / 4) + (g >> 2) * 8 + (g & 3)] = high;
          sh.q[b * (padded / 4) + (g >> 2) * 8 + 4 + (g & 3)] = low;
        }
      }
    }
  }

  // Vector memory of a compute unit returns in the order of its requests, whichever wavefront they
  // came from: no wavefront asks for weights before all of the workgroup have asked for their rows
  // (16384 -> 2048, one row: the last wavefront had its part of the row 3.4 us after the launch's
  // start behind the others' weights, now 2.8; the launch 8.0 -> 7.5 us).
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  // The ring: two tiles (18 KiB) per wavefront in flight. With several batch rows the second
  // tile is requested after the prologue's arithmetic, which then overlaps the time load issue
  // spends blocked on a full memory pipeline (measured: 15.4 -> 14.2 us at four rows); with one
  // row the prologue is too short for that to pay (9.0 -> 9.5 us), so both go out at once.
  constexpr int kRing = ALL > 0 ? ALL : kRingTiles;
  i32x4 ring[kRing][kPlanes];
  auto request_tile = [&](int t) {
    const int lin = min(kpart + t * ksplit, max(ntiles, 1) - 1);
    // The plane of scales goes first: loads return in issue order, so the rows of a tile can
    // then be worked through as they arrive instead of after the whole tile.
#pragma unroll
    for (int jj = 0; jj < kPlanes; ++jj) {
      const int j = (jj + kTileRows) % kPlanes;
      ring[t][j] =
          __builtin_nontemporal_load(tbase + static_cast<size_t>(lin) * kTileVecs + j * 64);
    }
  };
  constexpr int kPre = ALL > 0 ? PRE : (BT == 1 ? kRing : 1);
#pragma unroll
  for (int t = 0; t < kPre; ++t) request_tile(t);
  // Per-channel epilogue inputs of every channel this wavefront covers (lane = channel), parked in LDS
  // once the prologue is through. Their addresses come from the argument segment or the launch table:
  // asked for ahead of the rows, they held up every load of the launch by that read (start to first
  // load, with the division by ksplit: 0.45 us, now 0.2).
  const LRTFC_GLOBAL float* g_kfsum = (const LRTFC_GLOBAL float*)a.kfsum;
  const LRTFC_GLOBAL float* g_bias = (const LRTFC_GLOBAL float*)a.bias;
  LRTFC_GLOBAL float* g_output = (LRTFC_GLOBAL float*)a.output;
  const int my_n = min(first_group * kTileRows + lane, start.out_depth - 1);
  const float kfsum_raw = g_kfsum[my_n];
  const float bias_raw = a.bias ? g_bias[my_n] : 0.0f;
  __builtin_amdgcn_sched_barrier(0);
  // Chain lanes: lane = row * BT + batch.
  const int chain_row = lane / BT;
  const int chain_b = lane - chain_row * BT;
  const bool chain_lane = lane < kTileRows * BT;

  // This lane's row: its scale, multiplier and zero point.
  float row_scale = 0.0f, row_inv = 0.0f;
  int32_t row_zero_point = 0;

  // Activation rows into LDS.
  if (FUSED) {
    if (in_regs) {
#pragma unroll
      for (int b = 0; b < BT; ++b) {
        float mn = 0.0f, mx = 0.0f;
#pragma unroll
        for (int j = 0; j < kGroupsPerThread; ++j) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const float4 t = xr[b][j][h];  // clamped duplicates past the row are harmless here
            mn = fminf(fminf(mn, t.x), fminf(fminf(t.y, t.z), t.w));
            mx = fmaxf(fmaxf(mx, t.x), fmaxf(fmaxf(t.y, t.z), t.w));
          }
        }
        mn = WaveMinF32(mn);
        mx = WaveMaxF32(mx);
        if (lane == 0) {
          sh.mm[(b * kWaves + wave) * 2] = mn;
          sh.mm[(b * kWaves + wave) * 2 + 1] = mx;
        }
      }
    }
    __syncthreads();
    // Every wavefront derives the rows' parameters for itself, lane L those of row L % BT (the row whose
    // outputs a chain lane finishes): one barrier and a trip through LDS less than one lane doing it
    // for the workgroup (2048 -> 2048 at 1 / 4 rows 3.77 / 4.60 -> 3.63 / 4.41 us, 4096 -> 14336 at one
    // row 6.17 -> 6.02).
    {
      const int row = min(chain_b, bt - 1);
      float mn = sh.mm[row * kWaves * 2], mx = sh.mm[row * kWaves * 2 + 1];
#pragma unroll
      for (int w = 1; w < kWaves; ++w) {
        mn = fminf(mn, sh.mm[(row * kWaves + w) * 2]);
        mx = fmaxf(mx, sh.mm[(row * kWaves + w) * 2 + 1]);
      }
      const RowQuantParams qp = AsymmetricRowParams<VARIANT>(mn, mx);
      row_scale = qp.scale;
      row_inv = ElementwiseInv(qp);
      row_zero_point = qp.zero_point;
    }
    auto row_params = [&](int b) {
      RowQuantParams qp;
      qp.inv = ReadLaneF32(row_inv, b);
      qp.zero_point = __builtin_amdgcn_readlane(row_zero_point, b);
      return qp;
    };
    const int vector_end = depth - (depth % 8);
    if (in_regs) {
#pragma unroll
      for (int b = 0; b < BT; ++b) {
        if (b < bt) {
          const RowQuantParams qp = row_params(b);
#pragma unroll
          for (int j = 0; j < kGroupsPerThread; ++j) {
            const int g = j * kThreads + tid;
            if (g < padded / 8) {
              int32_t high = 0, low = 0;
              if (g < groups8) {
                const float4 lo = xr[b][j][0], hi = xr[b][j][1];
                const bool tail = g * 8 >= vector_end;
                NibblePlanes(
                    static_cast<uint32_t>(QuantizePack4<VARIANT>(lo.x, lo.y, lo.z, lo.w, qp, tail)),
                    static_cast<uint32_t>(QuantizePack4<VARIANT>(hi.x, hi.y, hi.z, hi.w, qp, tail)),
                    &high, &low);
              }
              sh.q[b * (padded / 4) + (g >> 2) * 8 + (g & 3)] = high;
              sh.q[b * (padded / 4) + (g >> 2) * 8 + 4 + (g & 3)] = low;
            }
          }
        }
      }
    } else {
      for (int b = 0; b < bt; ++b) {
        const LRTFC_GLOBAL float* x = g_input_f32 + static_cast<size_t>(batch0 + b) * depth;
        const RowQuantParams qp = row_params(b);
        for (int g = tid; g < padded / 8; g += kThreads) {
          int32_t v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
          if (g < groups8) {
            for (int t = 0; t < 8; ++t) {
              v[t] = QuantizeElement<VARIANT>(x[g * 8 + t], qp, true, g * 8 + t >= vector_end);
            }
          }
          int32_t high, low;
          NibblePlanes(static_cast<uint32_t>(PackBytes(v[0], v[1], v[2], v[3])),
                       static_cast<uint32_t>(PackBytes(v[4], v[5], v[6], v[7])), &high, &low);
          sh.q[b * (padded / 4) + (g >> 2) * 8 + (g & 3)] = high;
          sh.q[b * (padded / 4) + (g >> 2) * 8 + 4 + (g & 3)] = low;
        }
      }
    }
  } else if (in_regs) {
#pragma unroll
    for (int b = 0; b < BT; ++b) {
      if (b < bt) {
#pragma unroll
        for (int j = 0; j < kGroupsPerThread; ++j) {
          const int g = j * kThreads + tid;
          if (g < padded / 8) {
            int32_t high = 0, low = 0;
            if (g < groups8) {
              NibblePlanes(static_cast<uint32_t>(qr[b][j].x), static_cast<uint32_t>(qr[b][j].y),
                           &high, &low);
            }
            sh.q[b * (padded / 4) + (g >> 2) * 8 + (g & 3)] = high;
            sh.q[b * (padded / 4) + (g >> 2) * 8 + 4 + (g & 3)] = low;
          }
        }
      }
    }
  }
  __syncthreads();

#pragma unroll
  for (int t = kPre; t < kRing; ++t) request_tile(t);

  float* kb = sh.kb + wave * 2 * 64;
  kb[lane] = kfsum_raw;
  kb[64 + lane] = bias_raw;

  if (!FUSED && chain_lane && chain_b < bt) {
    row_scale = g_scaling_factors[batch0 + chain_b];
    row_zero_point = g_zero_points[batch0 + chain_b];
  }
  const float row_zp = static_cast<float>(row_zero_point);

  // Tile loop. Lane L owns block L of the tile for each of the 8 channels.
  constexpr int kTileFloats = 8 * BT * kPStride;
  float* pgroup = sh.p + static_cast<size_t>(group_in_wg) * chunks * kTileFloats;  // ksplit > 1
  float out = 0.0f;
  const int nblk = depth / kBlock;
  // One tile's 64 products per chain lane, added in block order.
  auto walk_tile = [&](const float* tile, int c) {
    const int count = min(kTileBlocks, nblk - c * kTileBlocks);
    const float* line = tile + lane * kPStride;
    if (count == kTileBlocks) {
      // Whole tile: fetch the 64 products with back-to-back LDS reads, then add in order.
      float4 v[kTileBlocks / 4];
#pragma unroll
      for (int j = 0; j < kTileBlocks / 4; ++j) v[j] = reinterpret_cast<const float4*>(line)[j];
#pragma unroll
      for (int j = 0; j < kTileBlocks / 4; ++j) {
        out = __fadd_rn(out, v[j].x);
        out = __fadd_rn(out, v[j].y);
        out = __fadd_rn(out, v[j].z);
        out = __fadd_rn(out, v[j].w);
      }
    } else {
      out = AddPartialTile(line, count, out);
    }
  };
  // fully_connected.cc:1078-1082 for the channel group at offset `goff` from the first. The
  // value is parked in LDS and leaves in one store at the end: a store inside the tile loop
  // would make the number of outstanding memory operations depend on the path taken, and
  // the waits for the ring would have to assume the worst.
  float* ob = sh.ob + wave * (kMaxGroupsPerWave * kTileRows * BT);
  auto finish_group = [&](int goff) {
    float o = __fsub_rn(out, __fmul_rn(row_zp, kb[goff * kTileRows + chain_row]));
    o = __fmul_rn(o, row_scale);
    if (a.bias) o = __fadd_rn(o, kb[64 + goff * kTileRows + chain_row]);
    ob[goff * kTileRows * BT + lane] = o;
  };
  // One tile: ring slot SLOT holds tile `lin` of this wavefront's stretch. REFILL requests the
  // tile two turns ahead into the same slot -- always, so that every turn of the main loop
  // issues the same number of loads and the wait for a slot can leave exactly the other slot's
  // loads in flight; past the end the request goes to one hot cache line instead.
  auto process = [&](auto slot_tag, auto refill_tag, int lin, int c) {
    constexpr int SLOT = decltype(slot_tag)::value;
    constexpr bool REFILL = decltype(refill_tag)::value;
    float* pw = ksplit == 1 ? sh.p + static_cast<size_t>(wave) * kTileFloats
                            : pgroup + static_cast<size_t>(c) * kTileFloats;
    // This block's activations (four dwords of high nibbles, four of low ones, per batch row)
    // and -8 * sum(low nibbles), the seed of the unsigned dot product.
    i32x4 qh[BT], ql[BT];
    uint32_t seed[BT];
    const int blk = c * kTileBlocks + lane;
#pragma unroll
    for (int b = 0; b < BT; ++b) {
      const i32x4* qp = reinterpret_cast<const i32x4*>(sh.q + b * (padded / 4) + blk * 8);
      qh[b] = qp[0];
      ql[b] = qp[1];
      uint32_t t = 0;
#pragma unroll
      for (int d = 0; d < 4; ++d) t = UDot8(static_cast<uint32_t>(ql[b][d]), 0x11111111u, t);
      seed[b] = 0u - 8u * t;
    }
    const i32x4 sc = ring[SLOT][kTileRows];
#pragma unroll
    for (int j = 0; j < kTileRows; ++j) {
      const uint32_t pair = static_cast<uint32_t>(sc[j >> 1]);
      const float scale =
          HalfBitsToFloatFast(static_cast<uint16_t>((j & 1) ? (pair >> 16) : (pair & 0xFFFF)));
      const i32x4 wv = ring[SLOT][j];  // nibbles stored as w + 8
      int32_t ws[4];                   // the same weights as signed nibbles
#pragma unroll
      for (int d = 0; d < 4; ++d) ws[d] = wv[d] ^ static_cast<int32_t>(0x88888888u);
#pragma unroll
      for (int b = 0; b < BT; ++b) {
        int32_t sd = 0;
        uint32_t ud = seed[b];
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          sd = SDot8(ws[d], qh[b][d], sd);
          ud = UDot8(static_cast<uint32_t>(wv[d]), static_cast<uint32_t>(ql[b][d]), ud);
        }
        const int32_t acc = (sd << 4) + static_cast<int32_t>(ud);
        pw[(j * BT + b) * kPStride + lane] = __fmul_rn(static_cast<float>(acc), scale);
      }
    }
    if (REFILL) {
      const int next = lin + kRingTiles * ksplit;
      const LRTFC_GLOBAL i32x4* src =
          next < ntiles ? tbase + static_cast<size_t>(next) * kTileVecs : g_packed;
#pragma unroll
      for (int jj = 0; jj < kPlanes; ++jj) {
        const int j = (jj + kTileRows) % kPlanes;
        ring[SLOT][j] = __builtin_nontemporal_load(src + j * 64);
      }
    }
    // Ordered float32 accumulation over this tile's blocks (same wavefront wrote them).
    if (ksplit == 1 && chain_lane) walk_tile(pw, c);
  };
  // Moves on to the next tile of the stretch; closes a channel group after its last tile.
#define LRTFC_INT4_ADVANCE()                      \
  do {                                            \
    if (ksplit == 1) {                            \
      if (++c == chunks) {                        \
        if (chain_lane) finish_group(goff);       \
        out = 0.0f;                               \
        c = 0;                                    \
        ++goff;                                   \
      }                                           \
    } else {                                      \
      c += ksplit;                                \
    }                                             \
  } while (0)
  int c = kpart;  // tile index within the current channel group
  int goff = 0;
  using Slot0 = std::integral_constant<int, 0>;
  using Slot1 = std::integral_constant<int, 1>;
  int lin = kpart;
  if constexpr (ALL > 0) {
    StaticFor<ALL>([&](auto t) {
      if (kpart + decltype(t)::value * ksplit < ntiles) {
        process(t, std::false_type{}, decltype(t)::value, c);
        LRTFC_INT4_ADVANCE();
      }
    });
  } else {
    for (; lin + ksplit < ntiles; lin += kRingTiles * ksplit) {
      process(Slot0{}, std::true_type{}, lin, c);
      LRTFC_INT4_ADVANCE();
      process(Slot1{}, std::true_type{}, lin + ksplit, c);
      LRTFC_INT4_ADVANCE();
    }
    if (lin < ntiles) {
      process(Slot0{}, std::false_type{}, lin, c);
      LRTFC_INT4_ADVANCE();
    }
  }
#undef LRTFC_INT4_ADVANCE
  if (ksplit > 1) {
    // Every tile of the group is parked; its first wavefront walks them in depth order.
    __syncthreads();
    if (kpart == 0 && chain_lane && my_groups > 0) {
      int cc = 0;
      if (ALL == 1 && nblk >= kTileBlocks) {
        cc = nblk / kTileBlocks;
        out = AddWholeTiles<kTileFloats>(pgroup + lane * kPStride, cc, out);
      }
      for (; cc < chunks; ++cc) walk_tile(pgroup + static_cast<size_t>(cc) * kTileFloats, cc);
      finish_group(0);
    }
  }
  // Outputs of this wavefront's channel groups: index = (group offset, row, batch).
  if (kpart == 0) {
    for (int i = lane; i < my_groups * kTileRows * BT; i += kWaveSize) {
      const int b = i % BT;
      const int row = i / BT;  // channel offset from the first group's first channel
      const int n = group0 * kTileRows + row;
      if (b < bt && n < start.out_depth) {
        g_output[static_cast<size_t>(batch0 + b) * start.out_depth + n] = ob[i];
      }
    }
  }
}

// The leading scalar arguments repeat what the first loads need (filter and row addresses,
// shapes): the library is built with kernel-argument preloading, which hands the leading scalar
// arguments to a wavefront in registers when it starts; the rest of the argument block is read
// from memory as usual while the first loads are already under way.
template <int BT, bool FUSED, int VARIANT, int GPT, int ALL, int PRE, int THREADS>
__global__ __launch_bounds__(THREADS) void FcInt4PackedKernel(
    const uint8_t* packed, const void* rows, int depth, int out_depth, int chunks, int batches,
    int batch0, int bt, int ksplit, int gpw, Int4PackedArgs rest) {
  extern __shared__ __align__(16) int8_t smem[];
  // Slices of the grid (gridDim.y > 1) take bt rows each, side by side.
  const int first_row = batch0 + static_cast<int>(blockIdx.y) * bt;
  FcInt4PackedBody<BT, FUSED, VARIANT, GPT, ALL, PRE, THREADS>(
      Int4Start{packed, rows, depth, out_depth, chunks}, rest, blockIdx.x, first_row,
      min(bt, batches - first_row), ksplit, gpw, smem);
}

// One channel group per workgroup on deep rows (DeepNode). Bound by latency: the additions of an output
// are a chain of one every 8 cycles, 1.8 us at 512 blocks, and behind the loads quantizing 16384 values
// and multiplying them takes as long again. Here eight wavefronts quantize and multiply in steps of two
// tiles, and a ninth adds a step's products while the others work on the next; in a step a wavefront has
// one tile's blocks of two channels, and everything is requested at the start. Filters not in the caches,
// us at 1 / 2 / 4 rows (4: int8 rows in, with their quantizer), FcInt4PackedKernel -> this one: 16384 ->
// 2048 8.7 / 10.7 / 14.1 -> 8.2 / 10.4 / 13.6, 11008 -> 2048 10.1 / 12.1 / 23.8 -> 7.5 / 9.7 / 12.0,
// 8192 -> 2048 6.4 / 8.1 / 11.2 -> 6.1 / 7.6 / 10.1, 4608 -> 1000 7.9 -> 5.0 at one row. A lane reads its
// two channels' scales alone: 92 registers at one row, with the whole plane 104 and 0.2 us more.
constexpr int kDeepWorkers = 8;
constexpr int kDeepThreads = (kDeepWorkers + 1) * kWaveSize;
constexpr int kDeepSteps = 4;  // of two tiles: depth up to 16384
constexpr int kStepTiles = 2;
constexpr int kWorkerThreads = kDeepWorkers * kWaveSize;  // eight values of a step each
static_assert(kWorkerThreads * 8 == kStepTiles * kTileBlocks * kBlock, "a step's values");

template <int BT>
constexpr size_t DeepLds(int chunks) {
  return static_cast<size_t>(BT) * chunks * kTileBlocks * kBlock +
         static_cast<size_t>(chunks) * kTileRows * BT * kPStride * 4 + BT * kDeepWorkers * 2 * 4;
}

template <int BT, bool FUSED, int VARIANT>
__global__ __launch_bounds__(kDeepThreads, 1) void FcInt4DeepKernel(
    const uint8_t* packed, const void* rows, int depth, int out_depth, int chunks, int batches,
    int batch0, int bt, Int4PackedArgs rest) {
  extern __shared__ __align__(16) int8_t smem[];
  const int tid = threadIdx.x;
  const int lane = tid & (kWaveSize - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWaveSize);
  const int padded = chunks * kTileBlocks * kBlock;
  const int steps = (chunks + kStepTiles - 1) / kStepTiles;
  const int group = blockIdx.x;
  int32_t* const q = reinterpret_cast<int32_t*>(smem);  // as in Int4Shared
  float* const p = reinterpret_cast<float*>(smem + static_cast<size_t>(BT) * padded);
  float* const mm = p + static_cast<size_t>(chunks) * kTileRows * BT * kPStride;  // [BT][workers][2]
  const int rows_here = min(bt, batches - batch0);
  const int b_here = lane & (BT - 1);  // the row whose parameters and outputs this lane has
  const int groups8 = depth / 8;

  // Every wavefront derives every row's parameters from the workers' ranges; lane L has row L % BT's.
  auto row_params = [&] {
    const int row = min(b_here, rows_here - 1);
    float mn = mm[row * kDeepWorkers * 2], mx = mm[row * kDeepWorkers * 2 + 1];
#pragma unroll
    for (int w = 1; w < kDeepWorkers; ++w) {
      mn = fminf(mn, mm[(row * kDeepWorkers + w) * 2]);
      mx = fmaxf(mx, mm[(row * kDeepWorkers + w) * 2 + 1]);
    }
    return AsymmetricRowParams<VARIANT>(mn, mx);
  };

  if (wave < kDeepWorkers) {
    // Rows, then (behind a barrier, see FcInt4PackedBody) weights.
    float4 xr[BT][kDeepSteps][2];
    i32x2 qr[BT][kDeepSteps];
#pragma unroll
    for (int b = 0; b < BT; ++b) {
      const size_t row = static_cast<size_t>(batch0 + min(b, rows_here - 1)) * depth;
#pragma unroll
      for (int j = 0; j < kDeepSteps; ++j) {
        const int g = min(j * kWorkerThreads + tid, groups8 - 1);
        if (FUSED) {
          const LRTFC_GLOBAL float* x = (const LRTFC_GLOBAL float*)rows + row + g * 8;
          const f32x4 lo = *reinterpret_cast<const LRTFC_GLOBAL f32x4*>(x);
          const f32x4 hi = *reinterpret_cast<const LRTFC_GLOBAL f32x4*>(x + 4);
          xr[b][j][0] = make_float4(lo.x, lo.y, lo.z, lo.w);
          xr[b][j][1] = make_float4(hi.x, hi.y, hi.z, hi.w);
        } else {
          qr[b][j] = *reinterpret_cast<const LRTFC_GLOBAL i32x2*>(
              (const LRTFC_GLOBAL int8_t*)rows + row + g * 8);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    const int half = wave >> 2, channel0 = 2 * (wave & 3);
    const LRTFC_GLOBAL i32x4* const tiles = (const LRTFC_GLOBAL i32x4*)packed +
                                            static_cast<size_t>(group) * chunks * kTileVecs + lane;
    i32x4 w[kDeepSteps][2];
    uint32_t sc[kDeepSteps];  // the two channels' scales, of the tile's last plane (eight a block)
#pragma unroll
    for (int j = 0; j < kDeepSteps; ++j) {
      const LRTFC_GLOBAL i32x4* tile = tiles + static_cast<size_t>(min(kStepTiles * j + half, chunks - 1)) * kTileVecs;
      sc[j] = ((const LRTFC_GLOBAL uint32_t*)(tile + kTileRows * 64))[channel0 / 2];
      w[j][0] = __builtin_nontemporal_load(tile + channel0 * 64);
      w[j][1] = __builtin_nontemporal_load(tile + (channel0 + 1) * 64);
    }
    __builtin_amdgcn_sched_barrier(0);
    float inv = 0.0f;
    int32_t zero_point = 0;
    if (FUSED) {
#pragma unroll
      for (int b = 0; b < BT; ++b) {
        float mn = 0.0f, mx = 0.0f;
#pragma unroll
        for (int j = 0; j < kDeepSteps; ++j) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const float4 t = xr[b][j][h];  // clamped duplicates past the row are harmless here
            mn = fminf(fminf(mn, t.x), fminf(fminf(t.y, t.z), t.w));
            mx = fmaxf(fmaxf(mx, t.x), fmaxf(fmaxf(t.y, t.z), t.w));
          }
        }
        mn = WaveMinF32(mn);
        mx = WaveMaxF32(mx);
        if (lane == 0) {
          mm[(b * kDeepWorkers + wave) * 2] = mn;
          mm[(b * kDeepWorkers + wave) * 2 + 1] = mx;
        }
      }
      __syncthreads();
      const RowQuantParams qp = row_params();
      inv = ElementwiseInv(qp);
      zero_point = qp.zero_point;
    }
#pragma unroll
    for (int j = 0; j < kDeepSteps; ++j) {
      if (j >= steps) break;
      const int g = j * kWorkerThreads + tid;
      if (g < padded / 8) {
#pragma unroll
        for (int b = 0; b < BT; ++b) {
          int32_t high = 0, low = 0;
          if (g < groups8) {
            uint32_t lo, hi;
            if (FUSED) {
              RowQuantParams qp;
              qp.inv = ReadLaneF32(inv, b);
              qp.zero_point = __builtin_amdgcn_readlane(zero_point, b);
              const float4 x0 = xr[b][j][0], x1 = xr[b][j][1];
              lo = static_cast<uint32_t>(QuantizePack4<VARIANT>(x0.x, x0.y, x0.z, x0.w, qp, /*tail=*/false));
              hi = static_cast<uint32_t>(QuantizePack4<VARIANT>(x1.x, x1.y, x1.z, x1.w, qp, /*tail=*/false));
            } else {
              lo = static_cast<uint32_t>(qr[b][j].x);
              hi = static_cast<uint32_t>(qr[b][j].y);
            }
            NibblePlanes(lo, hi, &high, &low);
          }
          q[b * (padded / 4) + (g >> 2) * 8 + (g & 3)] = high;
          q[b * (padded / 4) + (g >> 2) * 8 + 4 + (g & 3)] = low;
        }
      }
      __syncthreads();  // the step's rows are there, and the step before's products
      const int tile = kStepTiles * j + half;
      if (tile < chunks) {
        const int blk = tile * kTileBlocks + lane;
        const float scale[2] = {HalfBitsToFloatFast(static_cast<uint16_t>(sc[j] & 0xFFFF)),
                                HalfBitsToFloatFast(static_cast<uint16_t>(sc[j] >> 16))};
        i32x4 ws[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
#pragma unroll
          for (int d = 0; d < 4; ++d) ws[c][d] = w[j][c][d] ^ static_cast<int32_t>(0x88888888u);
        }
#pragma unroll
        for (int b = 0; b < BT; ++b) {
          const i32x4* at = reinterpret_cast<const i32x4*>(q + b * (padded / 4) + blk * 8);
          const i32x4 qh = at[0], ql = at[1];
          uint32_t t = 0;
#pragma unroll
          for (int d = 0; d < 4; ++d) t = UDot8(static_cast<uint32_t>(ql[d]), 0x11111111u, t);
          const uint32_t seed = 0u - 8u * t;
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            int32_t sd = 0;
            uint32_t ud = seed;
#pragma unroll
            for (int d = 0; d < 4; ++d) {
              sd = SDot8(ws[c][d], qh[d], sd);
              ud = UDot8(static_cast<uint32_t>(w[j][c][d]), static_cast<uint32_t>(ql[d]), ud);
            }
            const int32_t acc = (sd << 4) + static_cast<int32_t>(ud);
            p[((tile * kTileRows + channel0 + c) * BT + b) * kPStride + lane] =
                __fmul_rn(static_cast<float>(acc), scale[c]);
          }
        }
      }
    }
    __syncthreads();  // the last step's products
    return;
  }

  // The ninth wavefront: lane = channel * BT + row.
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_s_setprio(3);  // a chain of one addition at a time, the others fill what it leaves
  const int channel = min(group * kTileRows + lane / BT, out_depth - 1);
  const float kfsum = ((const LRTFC_GLOBAL float*)rest.kfsum)[channel];
  const float bias = rest.bias ? ((const LRTFC_GLOBAL float*)rest.bias)[channel] : 0.0f;
  float row_scale = 0.0f;
  int32_t row_zero_point = 0;
  if (FUSED) {
    __syncthreads();
    const RowQuantParams qp = row_params();
    row_scale = qp.scale;
    row_zero_point = qp.zero_point;
  } else {
    const int b = batch0 + min(b_here, rows_here - 1);
    row_scale = ((const LRTFC_GLOBAL float*)rest.scaling_factors)[b];
    row_zero_point = ((const LRTFC_GLOBAL int32_t*)rest.zero_points)[b];
  }
  const bool chain_lane = lane < kTileRows * BT;
  const int nblk = depth / kBlock;
  float out = 0.0f;
  constexpr int kTileFloats = kTileRows * BT * kPStride;
  auto add_step = [&](int j) {
    const float* line = p + static_cast<size_t>(kStepTiles * j) * kTileFloats + lane * kPStride;
    const int blocks = min(kStepTiles * kTileBlocks, nblk - kStepTiles * kTileBlocks * j);
    if (blocks == kStepTiles * kTileBlocks) {
      out = AddWholeTiles<kTileFloats>(line, kStepTiles, out);
    } else {
      const int whole = blocks / kTileBlocks;
      if (whole > 0) out = AddWholeTiles<kTileFloats>(line, whole, out);
      if (blocks % kTileBlocks) {
        out = AddPartialTile(line + static_cast<size_t>(whole) * kTileFloats, blocks % kTileBlocks, out);
      }
    }
  };
  for (int j = 0; j < steps; ++j) {
    __syncthreads();
    if (j > 0 && chain_lane) add_step(j - 1);
  }
  __syncthreads();
  if (chain_lane) {
    add_step(steps - 1);
    // fully_connected.cc:1078-1082
    float o = __fsub_rn(out, __fmul_rn(static_cast<float>(row_zero_point), kfsum));
    o = __fmul_rn(o, row_scale);
    if (rest.bias) o = __fadd_rn(o, bias);
    const int n = group * kTileRows + lane / BT;
    if (b_here < rows_here && n < out_depth) {
      ((LRTFC_GLOBAL float*)rest.output)[static_cast<size_t>(batch0 + b_here) * out_depth + n] = o;
    }
  }
}

// Several filters of the same depth in one launch (nodes of a graph that do not depend on
// each other: the q/k/v or gate/up projections of a decoder layer). The table lives in device
// memory: per node its arguments and the index of its first workgroup. One launch instead of
// `count` removes count - 1 launch gaps and lets small filters overlap large ones.
// Groups of up to kHeadNodes (q/k/v, gate/up) find their node and its first loads' addresses in the
// table's head, in one read; larger ones search first_block and read the node's arguments, three reads
// in sequence (a decoder of 6 layers of 1536 / 9216, one row, with the start above 195 -> 187 us).
constexpr int kHeadNodes = 4;
struct Int4GroupTable {
  int later_first[kHeadNodes];  // first workgroup of nodes 1, 2, 3 (INT32_MAX past the last)
  int out_depth[kHeadNodes];
  const void* rows[kHeadNodes];
  const uint8_t* packed[kHeadNodes];
  int first_block[kMaxGroupNodes + 1];
  int reserved[3];
  Int4PackedArgs node[kMaxGroupNodes];
};

template <int BT, bool FUSED, int VARIANT, int GPT, int ALL = 0, int PRE = 0, int THREADS = kThreads>
__global__ __launch_bounds__(THREADS) void FcInt4PackedGroupedKernel(
    const Int4GroupTable* __restrict__ table, int count, int depth, int chunks, int batches,
    int batch0, int bt, int ksplit, int gpw) {
  extern __shared__ __align__(16) int8_t smem[];
  const int block = blockIdx.x;
  Int4Start start;
  start.depth = depth;
  start.chunks = chunks;
  int node = 0, first = 0;
  if (count <= kHeadNodes) {
    start.rows = table->rows[0];
    start.packed = table->packed[0];
    start.out_depth = table->out_depth[0];
#pragma unroll
    for (int i = 1; i < kHeadNodes; ++i) {
      const int from = table->later_first[i - 1];
      const bool beyond = block >= from;
      node = beyond ? i : node;
      first = beyond ? from : first;
      start.rows = beyond ? table->rows[i] : start.rows;
      start.packed = beyond ? table->packed[i] : start.packed;
      start.out_depth = beyond ? table->out_depth[i] : start.out_depth;
    }
  } else {
    // first_block is ascending: the node of this workgroup is the number of later nodes whose
    // first workgroup is not beyond it. Vector loads and ballots (64 nodes per turn) instead of
    // a scalar walk.
    const int lane = threadIdx.x & (kWaveSize - 1);
    for (int base = 0; base + 1 < count; base += kWaveSize) {
      const int probe = base + lane + 1;
      const bool not_beyond = probe < count && block >= table->first_block[min(probe, count)];
      node += __popcll(__ballot(not_beyond));
    }
    node = __builtin_amdgcn_readfirstlane(node);
    first = table->first_block[node];
    start.rows = FUSED ? static_cast<const void*>(table->node[node].input_f32)
                       : static_cast<const void*>(table->node[node].input_q);
    start.packed = table->node[node].packed;
    start.out_depth = table->node[node].out_depth;
  }
  // Row tiles side by side (gridDim.y > 1): slice y of the grid takes rows batch0 + y * bt on.
  const int first_row = batch0 + static_cast<int>(blockIdx.y) * bt;
  FcInt4PackedBody<BT, FUSED, VARIANT, GPT, ALL, PRE, THREADS>(
      start, table->node[node], block - first, first_row, min(bt, batches - first_row), ksplit, gpw, smem);
}

// The row quantizer for a whole group: workgroup r quantizes row r % batches of node
// r / batches into that node's workspace (EvalBlockwise4Bit always quantizes asymmetrically,
// tflite/kernels/fully_connected.cc:1044-1047).
template <int VARIANT, int THREADS = kQuantizeThreads>
__global__ __launch_bounds__(THREADS) void QuantizeGroupRowsKernel(
    const Int4GroupTable* __restrict__ table, int batches) {
  const int node = blockIdx.x / batches;
  const int row = blockIdx.x - node * batches;
  const Int4PackedArgs& a = table->node[node];
  QuantizeRow<VARIANT, RowMajorPlacement, THREADS>(
                       a.input_f32 + static_cast<size_t>(row) * a.depth, a.depth,
                       const_cast<int8_t*>(a.input_q) + static_cast<size_t>(row) * a.depth, a.depth,
                       const_cast<float*>(a.scaling_factors) + row,
                       const_cast<int32_t*>(a.zero_points) + row, /*do_asymmetric=*/1);
}

// Depth up to 4096 keeps two groups per thread; up to 16384, eight. A fused launch holds
// the float rows (16 registers per group and row), so its deep form stops at two rows.
constexpr int kShallowGpt = 2;
constexpr int kShallowDepth = kShallowGpt * kThreads * 8;
constexpr int kDeepDepth = 8 * kThreads * 8;

// Wavefronts per channel group: one while that already gives the chip ~1000 wavefronts;
// otherwise the depth is shared out, as long as each wavefront keeps at least two tiles.
int ChooseKsplit(int out_depth, int chunks) {
  const int groups = (out_depth + kTileRows - 1) / kTileRows;
  int ksplit = 1;
  while (ksplit < kWaves && groups * ksplit < 1024 && chunks >= 4 * ksplit) ksplit *= 2;
  return ksplit;
}

// Single nodes of deep rows whose tiles make about one workgroup of eight wavefronts per CU, one tile
// each, beyond the groups of FcInt4DeepKernel (and unaligned rows within them): a wavefront alone on its
// SIMD issues a vector operation every 8 cycles or so, and the prologue (the row quantized and split into
// nibble planes by every workgroup) is the larger part of such a launch. Four wavefronts -> eight, us at
// 1 / 2 / 4 rows: 8192 -> 2048 8.3 / 9.7 / 13.4 -> 7.0 / 8.3 / 11.5. With two tiles each it is no gain
// (11008 -> 4096 11.1 -> 11.5 at one row), in more than one round a loss (4608 -> 12000 13.0 -> 17.3,
// 16384 -> 2050 14.4 -> 16.5).
bool WideDeep(int depth, int out_depth, int chunks) {
  constexpr int kWideWaves = kWideThreads / kWaveSize;
  if (depth <= kShallowDepth || depth > kDeepDepth) return false;
  if (chunks > kWideWaves || kWideWaves % chunks != 0) return false;
  const int groups = (out_depth + kTileRows - 1) / kTileRows;
  return groups <= kWideWaves / chunks * 256;
}

// Single nodes of deep rows with at most one channel group per CU: FcInt4DeepKernel. The rows have to
// lie on 16 bytes (8, as int8): the kernel has no other way to read them. Beyond one round of its
// workgroups every row is quantized once more per channel group than there: at one row 9216 -> 3072 9.5 ->
// 10.5 us, 8192 -> 4096 7.3 -> 10.0, 16384 -> 4096 13.3 -> 14.7.
constexpr int kDeepMaxGroups = 256;

bool DeepNode(const Int4PackedArgs& a, bool fused) {
  const auto at = reinterpret_cast<uintptr_t>(fused ? static_cast<const void*>(a.input_f32)
                                                    : static_cast<const void*>(a.input_q));
  return a.depth > kShallowDepth && a.depth <= kDeepDepth && (at & (fused ? 15 : 7)) == 0 &&
         (a.out_depth + kTileRows - 1) / kTileRows <= kDeepMaxGroups;
}

// Channel groups per wavefront. Measured on launches from 7 MB to 340 MB: a wavefront should
// stream up to 8 tiles (its ring then runs long enough to amortize the prologue), as long as
// the launch keeps about one workgroup per CU (224 of them) to spread over the chip.
int ChooseGroupsPerWave(int total_groups, int chunks, int ksplit) {
  if (ksplit > 1) return 1;
  int gpw = 1;
  while (gpw * 2 <= kMaxGroupsPerWave && gpw * 2 * chunks <= 8 &&
         total_groups / (kWaves * gpw * 2) >= 224) {
    gpw *= 2;
  }
  return gpw;
}

template <int BT, bool FUSED, int VARIANT, int GPT, int ALL, int PRE, int THREADS = kThreads>
hipError_t LaunchSized(const Int4PackedArgs& a, int batch0, int bt, int slices, int ksplit, int gpw,
                       hipStream_t stream) {
  const int padded = a.chunks * kTileBlocks * kBlock;
  const size_t lds = Int4Shared<BT, THREADS>::Bytes(padded, ksplit);
  auto kernel = FcInt4PackedKernel<BT, FUSED, VARIANT, GPT, ALL, PRE, THREADS>;
  if (hipError_t err = EnsureDynamicLds(reinterpret_cast<const void*>(kernel), lds)) return err;
  const int groups = (a.out_depth + kTileRows - 1) / kTileRows;
  const int groups_per_wg = THREADS / kWaveSize / ksplit * gpw;
  const int grid = (groups + groups_per_wg - 1) / groups_per_wg;
  const void* rows = FUSED ? static_cast<const void*>(a.input_f32) : static_cast<const void*>(a.input_q);
  hipLaunchKernelGGL(kernel, dim3(grid, slices), dim3(THREADS), lds, stream, a.packed, rows, a.depth,
                     a.out_depth, a.chunks, a.batches, batch0, bt, ksplit, gpw, a);
  return hipGetLastError();
}

// A single node of up to two batch rows whose wavefronts can be given at most two tiles each
// (depth up to 4096) runs the straight-line form: first tile ahead of the prologue, second
// behind it.
constexpr int kStraightTiles = 2;

template <int BT, bool FUSED, int VARIANT, int GPT>
hipError_t LaunchOne(const Int4PackedArgs& a, int batch0, int bt, int slices, hipStream_t stream) {
  if constexpr (GPT > kShallowGpt) {
    if (DeepNode(a, FUSED)) {
      const size_t lds = DeepLds<BT>(a.chunks);
      auto kernel = FcInt4DeepKernel<BT, FUSED, VARIANT>;
      if (hipError_t err = EnsureDynamicLds(reinterpret_cast<const void*>(kernel), lds)) return err;
      const void* rows = FUSED ? static_cast<const void*>(a.input_f32) : static_cast<const void*>(a.input_q);
      hipLaunchKernelGGL(kernel, dim3((a.out_depth + kTileRows - 1) / kTileRows), dim3(kDeepThreads), lds,
                         stream, a.packed, rows, a.depth, a.out_depth, a.chunks, a.batches, batch0, bt, a);
      return hipGetLastError();
    }
    if (WideDeep(a.depth, a.out_depth, a.chunks)) {
      return LaunchSized<BT, FUSED, VARIANT, GPT * kThreads / kWideThreads, 1, 1, kWideThreads>(
          a, batch0, bt, slices, /*ksplit=*/a.chunks, 1, stream);
    }
  }
  const int ksplit = ChooseKsplit(a.out_depth, a.chunks);
  const int groups = (a.out_depth + kTileRows - 1) / kTileRows;
  int gpw = ChooseGroupsPerWave(groups, a.chunks, ksplit);
  if constexpr (BT <= 2) {
    if (ksplit == 1 && a.chunks <= kStraightTiles) {
      gpw = min(gpw, kStraightTiles / a.chunks);
      return LaunchSized<BT, FUSED, VARIANT, GPT, kStraightTiles, 1>(a, batch0, bt, slices, ksplit,
                                                                     gpw, stream);
    }
  }
  return LaunchSized<BT, FUSED, VARIANT, GPT, 0, 0>(a, batch0, bt, slices, ksplit, gpw, stream);
}

template <int BT, bool FUSED, int GPT>
hipError_t LaunchVariant(const Int4PackedArgs& a, int variant, int batch0, int bt, int slices,
                         hipStream_t stream) {
  if constexpr (!FUSED) {
    return LaunchOne<BT, false, LRTFC_QUANT_PORTABLE, GPT>(a, batch0, bt, slices, stream);
  } else {
    switch (variant) {
    case LRTFC_QUANT_NEON_V8:
      return LaunchOne<BT, FUSED, LRTFC_QUANT_NEON_V8, GPT>(a, batch0, bt, slices, stream);
    case LRTFC_QUANT_NEON_LEGACY:
      return LaunchOne<BT, FUSED, LRTFC_QUANT_NEON_LEGACY, GPT>(a, batch0, bt, slices, stream);
    default:
      return LaunchOne<BT, FUSED, LRTFC_QUANT_PORTABLE, GPT>(a, batch0, bt, slices, stream);
  }
  }
}

template <bool FUSED>
int MaxBatchTile(int depth) {
  return (FUSED && depth > kShallowDepth && depth <= kDeepDepth) ? 2 : 4;
}

// A workgroup may use 160 KB of LDS; the maps below keep 10 KB clear of that.
constexpr size_t kLdsBudget = 150 * 1024;

// Rows per launch: `want` (1, 2 or 4) cut down until the LDS map of that many rows fits.
int FitBatchTile(int want, int padded, int ksplit, bool wide = false) {
  int bt = want > 2 ? 4 : want;
  auto bytes = [&](int rows) {
    if (wide) {
      return rows > 2 ? Int4Shared<4, kWideThreads>::Bytes(padded, ksplit)
                      : Int4Shared<2, kWideThreads>::Bytes(padded, ksplit);
    }
    return rows > 2 ? Int4Shared<4>::Bytes(padded, ksplit) : Int4Shared<2>::Bytes(padded, ksplit);
  };
  while (bt > 1 && bytes(bt) > kLdsBudget) bt = bt > 2 ? 2 : 1;
  return bt;
}

static_assert(DeepLds<4>(kDeepSteps * kStepTiles) <= kLdsBudget, "four deep rows fit whatever their depth");

// Rows of a launch of a single node, by the LDS map of the kernel that LaunchOne takes.
int RowsPerLaunch(const Int4PackedArgs& a, bool fused) {
  const int most = fused ? MaxBatchTile<true>(a.depth) : MaxBatchTile<false>(a.depth);
  if (DeepNode(a, fused)) return most;
  const bool wide = WideDeep(a.depth, a.out_depth, a.chunks);
  return FitBatchTile(most, a.chunks * kTileBlocks * kBlock,
                      wide ? a.chunks : ChooseKsplit(a.out_depth, a.chunks), wide);
}

template <bool FUSED>
hipError_t LaunchTile(const Int4PackedArgs& a, int variant, int batch0, int bt, int slices,
                      hipStream_t stream) {
  if (a.depth > kShallowDepth && a.depth <= kDeepDepth) {
    if (bt <= 1) return LaunchVariant<1, FUSED, 8>(a, variant, batch0, bt, slices, stream);
    if (bt <= 2) return LaunchVariant<2, FUSED, 8>(a, variant, batch0, bt, slices, stream);
    if (!FUSED) return LaunchVariant<4, false, 8>(a, variant, batch0, bt, slices, stream);
    return hipErrorInvalidValue;  // MaxBatchTile keeps fused deep launches at two rows
  }
  if (bt <= 1) return LaunchVariant<1, FUSED, 2>(a, variant, batch0, bt, slices, stream);
  if (bt <= 2) return LaunchVariant<2, FUSED, 2>(a, variant, batch0, bt, slices, stream);
  return LaunchVariant<4, FUSED, 2>(a, variant, batch0, bt, slices, stream);
}

}  // namespace

size_t PackedInt4BlockwiseBytes(int out_depth, int depth) {
  const size_t groups = (static_cast<size_t>(out_depth) + kTileRows - 1) / kTileRows;
  const size_t chunks = (static_cast<size_t>(depth) / kBlock + kTileBlocks - 1) / kTileBlocks;
  return groups * chunks * kTileBytes;
}

hipError_t LaunchPackInt4Blockwise(const uint8_t* filter, const uint16_t* scales, int out_depth,
                                   int depth, uint8_t* packed, hipStream_t stream) {
  if (out_depth == 0 || depth == 0) return hipSuccess;
  const int chunks = (depth / kBlock + kTileBlocks - 1) / kTileBlocks;
  const int64_t total_vecs = static_cast<int64_t>(PackedInt4BlockwiseBytes(out_depth, depth) / 16);
  const unsigned grid = static_cast<unsigned>((total_vecs + kThreads - 1) / kThreads);
  hipLaunchKernelGGL(PackInt4BlockwiseKernel, dim3(grid), dim3(kThreads), 0, stream, filter,
                     scales, out_depth, depth, chunks, total_vecs, packed);
  return hipGetLastError();
}

bool FcInt4PackedSupports(int depth, int blocksize) {
  if (blocksize != kBlock || depth <= 0 || depth % kBlock != 0) return false;
  const int chunks = (depth / kBlock + kTileBlocks - 1) / kTileBlocks;
  return Int4Shared<1>::Bytes(chunks * kTileBlocks * kBlock, kWaves) <= kLdsBudget;
}

hipError_t LaunchFcInt4Packed(const FcInt4Args& q, const uint8_t* packed, const float* input_f32,
                              int variant, hipStream_t stream) {
  if (q.batches == 0 || q.out_depth == 0) return hipSuccess;
  if (!FcInt4PackedSupports(q.depth, q.blocksize)) return hipErrorNotSupported;
  Int4PackedArgs a;
  a.packed = packed;
  a.input_f32 = input_f32;
  a.input_q = q.input;
  a.scaling_factors = q.scaling_factors;
  a.zero_points = q.zero_points;
  a.kfsum = q.kfsum;
  a.bias = q.bias;
  a.output = q.output;
  a.batches = q.batches;
  a.depth = q.depth;
  a.out_depth = q.out_depth;
  a.chunks = (q.depth / kBlock + kTileBlocks - 1) / kTileBlocks;
  // Three or four fused rows of a small filter: two pairs side by side in one launch, as in small
  // groups (PrepareInt4Group); us at four rows, one tile of four -> pairs: 2048 -> 2048 6.8 -> 4.8,
  // 4096 -> 4096 8.7 -> 6.0. Both slices together are one round of a workgroup per CU; in two they read
  // the filter from memory twice (filters not in the cache: 2976 -> 5003 9.0 -> 10.0, 2976 -> 8192
  // 9.2 -> 9.9, 4096 -> 7700 9.2 -> 9.9; in it, 2048 -> 8192 6.9 -> 6.3).
  if (input_f32 && (q.batches == 3 || q.batches == 4) && q.depth <= kShallowDepth &&
      static_cast<int64_t>(q.out_depth) * q.depth / 2 <= kSideBySideMaxFilterBytes) {
    const int groups_per_wg = kWaves / ChooseKsplit(q.out_depth, a.chunks);
    const int blocks = ((q.out_depth + kTileRows - 1) / kTileRows + groups_per_wg - 1) / groups_per_wg;
    if (2 * blocks <= kPairRound) return LaunchTile<true>(a, variant, 0, 2, 2, stream);
  }
  const int tile = RowsPerLaunch(a, input_f32 != nullptr);
  int batch0 = 0;
  while (batch0 < q.batches) {
    const int bt = min(tile, q.batches - batch0);
    const hipError_t err = input_f32 ? LaunchTile<true>(a, variant, batch0, bt, 1, stream)
                                     : LaunchTile<false>(a, variant, batch0, bt, 1, stream);
    if (err != hipSuccess) return err;
    batch0 += bt;
  }
  return hipSuccess;
}

int FcInt4PackedRowsPerLaunch(int depth, int out_depth, bool fused) {
  Int4PackedArgs a{};  // null pointers: aligned ones
  a.depth = depth;
  a.out_depth = out_depth;
  a.chunks = (depth / kBlock + kTileBlocks - 1) / kTileBlocks;
  return RowsPerLaunch(a, fused);
}

hipError_t PrepareInt4Group(const lrtfc_int4_group_node* nodes, int count, int batches, int depth,
                            void* device_table, lrtfc_int4_group_launch* launch,
                            hipStream_t stream) {
  if (count < 1 || count > kMaxGroupNodes || !FcInt4PackedSupports(depth, kBlock)) {
    return hipErrorInvalidValue;
  }
  if (batches < 1) return hipErrorInvalidValue;
  {
    int total_tiles = 0;
    for (int i = 0; i < count; ++i) total_tiles += (nodes[i].out_depth + 15) / 16;
    bool nibbles = Int4NibbleGroupWins(batches, depth, total_tiles);
    bool decode = true;
    for (int i = 0; i < count; ++i) {
      nibbles = nibbles && nodes[i].nibble_filter != nullptr && nodes[i].workspace != nullptr;
      decode = decode && nodes[i].retiled_filter != nullptr;
    }
    if (nibbles) {
      return PrepareInt4NibbleGroup(nodes, count, batches, depth, device_table, launch, stream);
    }
    if (!decode) return hipErrorInvalidValue;
  }
  const int chunks = (depth / kBlock + kTileBlocks - 1) / kTileBlocks;
  int total_out = 0;
  for (int i = 0; i < count; ++i) total_out += nodes[i].out_depth;
  const int ksplit = ChooseKsplit(total_out, chunks);
  const int gpw = ChooseGroupsPerWave((total_out + kTileRows - 1) / kTileRows, chunks, ksplit);
  const int groups_per_wg = kWaves / ksplit * gpw;
  // Deep rows keep at most two in registers through the fused prologue; more rows are
  // quantized by a launch of their own when every node has a workspace to receive them.
  // Shallow rows do the same only in launches of many workgroups, where quantizing each row
  // once instead of once per workgroup outweighs the extra launch (config 5, B = 4: the 108
  // nodes of depth 2048 in 272 instead of 280 us per token; groups of one to three nodes lose).
  int total_blocks = 0;
  for (int i = 0; i < count; ++i) {
    const int groups = (nodes[i].out_depth + kTileRows - 1) / kTileRows;
    total_blocks += (groups + groups_per_wg - 1) / groups_per_wg;
  }
  bool split = batches > 2 && depth <= kDeepDepth &&
               (depth > kShallowDepth || total_blocks >= kSplitShallowMinBlocks);
  for (int i = 0; i < count; ++i) split = split && nodes[i].workspace != nullptr;
  // Three or four rows of a SMALL group (a stage of a decoder: one to three nodes that leave
  // most of the chip without a workgroup, their filters a few megabytes that the second reader
  // finds in the caches): the rows go as two pairs side by side in ONE launch, each workgroup
  // quantizing and multiplying two rows (2048 x 2048 at four rows: 6.3 us as one tile of four,
  // 4.7 us for two rows; 2048 x 16384: 16.5 us with the quantizer launch, 12.0 us for two fused
  // rows). Larger filters lose: the two 2048 -> 16384 projections of a decoder layer, 33.5 MB,
  // as pairs side by side take config 5's decoder-ordered token from 688 to 736 us.
  const int64_t filter_bytes = static_cast<int64_t>(total_out) * depth / 2;
  const bool side_by_side = (batches == 3 || batches == 4) && depth <= kDeepDepth &&
                            total_blocks <= kSideBySideMaxBlocks &&
                            filter_bytes <= kSideBySideMaxFilterBytes &&
                            FitBatchTile(2, chunks * kTileBlocks * kBlock, ksplit) == 2;
  if (side_by_side) split = false;
  Int4GroupTable host{};
  int next = 0;
  for (int i = 0; i < count; ++i) {
    host.first_block[i] = next;
    Int4PackedArgs& a = host.node[i];
    a.packed = nodes[i].retiled_filter;
    a.input_f32 = nodes[i].input;
    a.input_q = nullptr;
    a.scaling_factors = nullptr;
    a.zero_points = nullptr;
    if (split) {
      const ActivationWorkspace w = SplitActivationWorkspace(nodes[i].workspace, batches, depth);
      a.input_q = w.q;
      a.scaling_factors = w.sf;
      a.zero_points = w.zp;
    }
    a.kfsum = nodes[i].kfsum;
    a.bias = nodes[i].bias;
    a.output = nodes[i].output;
    a.batches = batches;
    a.depth = depth;
    a.out_depth = nodes[i].out_depth;
    a.chunks = chunks;
    const int groups = (nodes[i].out_depth + kTileRows - 1) / kTileRows;
    next += (groups + groups_per_wg - 1) / groups_per_wg;
  }
  host.first_block[count] = next;
  for (int i = 0; i < kHeadNodes; ++i) {
    const Int4PackedArgs& a = host.node[min(i, count - 1)];
    host.out_depth[i] = a.out_depth;
    host.rows[i] = split ? static_cast<const void*>(a.input_q) : static_cast<const void*>(a.input_f32);
    host.packed[i] = a.packed;
    host.later_first[i] = i + 1 < count ? host.first_block[i + 1] : INT32_MAX;
  }
  // Synchronous: the table is a stack object.
  hipError_t err = hipMemcpyAsync(device_table, &host, sizeof(host), hipMemcpyHostToDevice, stream);
  if (err == hipSuccess) err = hipStreamSynchronize(stream);
  if (err != hipSuccess) return err;
  launch->count = count;
  launch->grid_blocks = next;
  launch->ksplit = ksplit;
  launch->groups_per_wave = gpw;
  launch->batches = batches;
  launch->depth = depth;
  launch->split_quantize = side_by_side ? kRowPairsSideBySide : (split ? 1 : 0);
  launch->form = LRTFC_INT4_FORM_DECODE;
  return hipSuccess;
}

size_t Int4GroupTableBytes() {
  return sizeof(Int4GroupTable) > Int4NibbleGroupTableBytes() ? sizeof(Int4GroupTable)
                                                              : Int4NibbleGroupTableBytes();
}

namespace {
template <int BT, bool FUSED, int VARIANT, int GPT, int ALL = 0, int PRE = 0, int THREADS = kThreads>
hipError_t LaunchGroupedOne(const void* table, const lrtfc_int4_group_launch& l, int batch0,
                            int bt, hipStream_t stream, int row_tiles = 1) {
  const int chunks = (l.depth / kBlock + kTileBlocks - 1) / kTileBlocks;
  const int padded = chunks * kTileBlocks * kBlock;
  const size_t lds = Int4Shared<BT, THREADS>::Bytes(padded, l.ksplit);
  auto kernel = FcInt4PackedGroupedKernel<BT, FUSED, VARIANT, GPT, ALL, PRE, THREADS>;
  if (hipError_t err = EnsureDynamicLds(reinterpret_cast<const void*>(kernel), lds)) return err;
  hipLaunchKernelGGL(kernel, dim3(l.grid_blocks, row_tiles), dim3(THREADS), lds, stream,
                     static_cast<const Int4GroupTable*>(table), l.count, l.depth, chunks, l.batches,
                     batch0, bt, l.ksplit, l.groups_per_wave * kThreads / THREADS);
  return hipGetLastError();
}

template <int BT, int GPT, int ALL = 0, int PRE = 0, int THREADS = kThreads>
hipError_t LaunchGroupedVariant(const void* table, const lrtfc_int4_group_launch& l, int variant,
                                int batch0, int bt, hipStream_t stream, int row_tiles = 1) {
  switch (variant) {
    case LRTFC_QUANT_NEON_V8:
      return LaunchGroupedOne<BT, true, LRTFC_QUANT_NEON_V8, GPT, ALL, PRE, THREADS>(
          table, l, batch0, bt, stream, row_tiles);
    case LRTFC_QUANT_NEON_LEGACY:
      return LaunchGroupedOne<BT, true, LRTFC_QUANT_NEON_LEGACY, GPT, ALL, PRE, THREADS>(
          table, l, batch0, bt, stream, row_tiles);
    default:
      return LaunchGroupedOne<BT, true, LRTFC_QUANT_PORTABLE, GPT, ALL, PRE, THREADS>(
          table, l, batch0, bt, stream, row_tiles);
  }
}

hipError_t LaunchGroupQuantizer(const void* table, const lrtfc_int4_group_launch& l, int variant,
                                hipStream_t stream) {
  const auto* t = static_cast<const Int4GroupTable*>(table);
  const dim3 grid(static_cast<unsigned>(l.count) * l.batches);
  const bool deep = l.depth > kQuantizeDeepRow;
  auto launch = [&](auto narrow, auto wide) {
    if (deep) {
      hipLaunchKernelGGL(wide, grid, dim3(kQuantizeDeepThreads), 0, stream, t, l.batches);
    } else {
      hipLaunchKernelGGL(narrow, grid, dim3(kQuantizeThreads), 0, stream, t, l.batches);
    }
  };
  switch (variant) {
    case LRTFC_QUANT_NEON_V8:
      launch(QuantizeGroupRowsKernel<LRTFC_QUANT_NEON_V8>,
             QuantizeGroupRowsKernel<LRTFC_QUANT_NEON_V8, kQuantizeDeepThreads>);
      break;
    case LRTFC_QUANT_NEON_LEGACY:
      launch(QuantizeGroupRowsKernel<LRTFC_QUANT_NEON_LEGACY>,
             QuantizeGroupRowsKernel<LRTFC_QUANT_NEON_LEGACY, kQuantizeDeepThreads>);
      break;
    default:
      launch(QuantizeGroupRowsKernel<LRTFC_QUANT_PORTABLE>,
             QuantizeGroupRowsKernel<LRTFC_QUANT_PORTABLE, kQuantizeDeepThreads>);
      break;
  }
  return hipGetLastError();
}
}  // namespace

hipError_t LaunchFcInt4PackedGrouped(const void* table, const lrtfc_int4_group_launch& l,
                                     int variant, hipStream_t stream) {
  if (l.count < 1 || l.grid_blocks < 1) return hipSuccess;
  if (l.form == LRTFC_INT4_FORM_GEMM_NIBBLES) {
    return LaunchFcInt4NibbleGrouped(table, l, variant, stream);
  }
  const int chunks = (l.depth / kBlock + kTileBlocks - 1) / kTileBlocks;
  const int padded = chunks * kTileBlocks * kBlock;
  if (l.split_quantize == 1) {
    if (hipError_t err = LaunchGroupQuantizer(table, l, variant, stream)) return err;
    const bool deep_rows = l.depth > kShallowDepth;
    const int tile = FitBatchTile(4, padded, l.ksplit);
    for (int batch0 = 0; batch0 < l.batches; batch0 += tile) {
      const int bt = min(tile, l.batches - batch0);
      hipError_t err;
      if (deep_rows) {
        err = bt <= 1   ? LaunchGroupedOne<1, false, LRTFC_QUANT_PORTABLE, 8>(table, l, batch0, bt, stream)
              : bt <= 2 ? LaunchGroupedOne<2, false, LRTFC_QUANT_PORTABLE, 8>(table, l, batch0, bt, stream)
                        : LaunchGroupedOne<4, false, LRTFC_QUANT_PORTABLE, 8>(table, l, batch0, bt, stream);
      } else {
        err = bt <= 1   ? LaunchGroupedOne<1, false, LRTFC_QUANT_PORTABLE, 2>(table, l, batch0, bt, stream)
              : bt <= 2 ? LaunchGroupedOne<2, false, LRTFC_QUANT_PORTABLE, 2>(table, l, batch0, bt, stream)
                        : LaunchGroupedOne<4, false, LRTFC_QUANT_PORTABLE, 2>(table, l, batch0, bt, stream);
      }
      if (err != hipSuccess) return err;
    }
    return hipSuccess;
  }
  const bool deep = l.depth > kShallowDepth && l.depth <= kDeepDepth;
  if (l.split_quantize == kRowPairsSideBySide) {
    // Three or four rows of a small group: two slices of the grid, two fused rows each.
    return deep ? LaunchGroupedVariant<2, 8>(table, l, variant, 0, 2, stream, 2)
                : LaunchGroupedVariant<2, 2>(table, l, variant, 0, 2, stream, 2);
  }
  // One row, and the tiles of a wavefront known: straight-line code, as for single nodes. One tile each:
  // 2048 -> 2048 + 256 + 256 4.75 -> 4.2 us, 1152 -> 6912 + 6912 8.7 -> 7.2. Four each (beyond that a group
  // fills the ring's turns): eight wavefronts a workgroup with two each, one ahead of the prologue: 2048 ->
  // 2 x 16384 9.45 -> 9.0 us, 4096 -> 2 x 11008 13.9 -> 13.4, 2048 -> 18 x 2048 13.4 -> 12.5 (both ahead, or
  // both behind: 10). Two each stay with the ring, which requests both ahead: straight-line 2 % slower. So
  // do two and more rows, where neither form is a gain (6 layers of 2048 / 12288 at two rows 175.5 us a
  // token, with both 176.5).
  if (l.batches == 1 && l.depth <= kShallowDepth && l.ksplit == 1) {
    const int tiles = l.groups_per_wave * chunks;
    if (tiles == 1) return LaunchGroupedVariant<1, kShallowGpt, 1, 1>(table, l, variant, 0, 1, stream);
    if (tiles == 2 * kStraightTiles && l.groups_per_wave % 2 == 0) {
      return LaunchGroupedVariant<1, kShallowGpt * kThreads / kWideThreads, kStraightTiles, 1, kWideThreads>(
          table, l, variant, 0, 1, stream);
    }
  }
  const int tile = FitBatchTile(MaxBatchTile<true>(l.depth), padded, l.ksplit);
  for (int batch0 = 0; batch0 < l.batches; batch0 += tile) {  // more rows: one launch per tile
    const int bt = min(tile, l.batches - batch0);
    hipError_t err;
    if (deep) {
      err = bt <= 1 ? LaunchGroupedVariant<1, 8>(table, l, variant, batch0, bt, stream)
                    : LaunchGroupedVariant<2, 8>(table, l, variant, batch0, bt, stream);
    } else if (bt <= 1) {
      err = LaunchGroupedVariant<1, 2>(table, l, variant, batch0, bt, stream);
    } else if (bt <= 2) {
      err = LaunchGroupedVariant<2, 2>(table, l, variant, batch0, bt, stream);
    } else {
      err = LaunchGroupedVariant<4, 2>(table, l, variant, batch0, bt, stream);
    }
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

}  // namespace lrtfc
