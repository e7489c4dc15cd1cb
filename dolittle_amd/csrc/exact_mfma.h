// Exact many-row projections on the FP32 matrix cores.
//
// The reference projection (src/kernels/cuda/projection.cu:139-482) fixes, for
// every (row, output), P strided partial sums: partial t is the FMA chain over
// inputs t, t + P, ... in ascending order, merged upper into lower at offsets
// P/2..1.  An FP32 MFMA of depth 1 (v_mfma_f32_32x32x1_2b_f32) is one such FMA
// per element: D = A B + C with a single rounding, to nearest even, subnormals
// kept (on MI355X equal bit for bit to fmaf on 0.4 million random, subnormal
// and infinite operands per shape).  Its two independent 32 x 32 blocks hold
// two partials of the same 32 outputs x 32 rows, so P / 2 instructions advance
// all P chains by one input each, with the chains' order and merge untouched.
//
// The matrix cores run FP32 at twice the FMA rate of the vector ALUs without
// packed instructions: 67-75 T FMA/s measured against 39-51.  Vector
// instructions of either wavefront of a SIMD do not overlap with them (about 4
// clocks each), so what counts is how few widenings a product needs: two per
// 32 x 32 x 2 products here (66 T FMA/s in isolation), against 1.5 per 16 x 16
// x 4 with two row tiles per wavefront (50 T FMA/s for the 512-row gate/up).
//
// Operand orders.  A stage holds 8 chain steps (8 P inputs) of every row, in
// 16-byte pieces.  Permuted rows (the packed weights, the P-permuted
// activations) keep 8 consecutive elements of one chain in a piece: piece t is
// chain t.  Natural rows (row-major weights) keep 8 consecutive inputs: input
// P e + t of step e lies in piece (P e + t) / 8.
#pragma once

#include "dl_device.h"

namespace dl::exact {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x32 __attribute__((ext_vector_type(32)));

enum class Order { kPermuted, kNatural };

// A workgroup computes TM x TN tiles of Edge outputs x Edge rows (32, or 16
// with the four-block v_mfma_f32_16x16x1_4b_f32 where there are few rows);
// Split wavefronts share a tile, each with P / Split of its chains.  Block b
// of instruction w of wavefront c holds chain t = (P / Blocks) b + Split w + c,
// so the offsets P/2 .. Split merge inside a lane and only the last
// log2(Split) offsets cross wavefronts.  A stage is Groups x 8 chain steps.
template <int P_, int Edge_, int Split_, int TM_, int TN_, int Groups_, int Ring_, Order Weights_, Order Rows_>
struct Tile {
  static constexpr int P = P_, Edge = Edge_, Split = Split_, TM = TM_, TN = TN_, kGroups = Groups_, kRing = Ring_;
  static constexpr Order kWeights = Weights_, kRowOrder = Rows_;
  static constexpr int kBlocks = 64 / Edge, kChains = P / kBlocks;  // chains per block
  static constexpr int W = kChains / Split;                         // instructions per chain step
  static constexpr int kWaves = TM * TN * Split, kThreads = 64 * kWaves;
  static constexpr int kOutputs = Edge * TM, kRows = Edge * TN;
  static constexpr int kStageRows = kOutputs + kRows;
  static constexpr int kPieces = kGroups * P, kRowBytes = 16 * kPieces;  // per stage row
  static constexpr int kInputs = 8 * kPieces;                            // inputs per stage
  static constexpr int kLoads = kStageRows * kPieces / 64 / kWaves;      // 1 KiB loads per wavefront and stage
  static constexpr int kStageBytes = kStageRows * kRowBytes;
  static constexpr int kRegs = 1024 / 64 * (Edge == 32 ? 2 : 1);  // accumulators per instruction
  static_assert((Edge == 32 || Edge == 16) && (P == 16 || P == 32) && W >= 1 && kChains % Split == 0, "tile shape");
  static_assert(kStageRows * kPieces % (64 * kWaves) == 0, "whole loads per wavefront");
  static_assert(kRing >= 2 && kRing <= 4, "two to four stage buffers");
};

// Rows up to which 16-row tiles beat 32-row ones: they give four times the
// workgroups and waste less on a remainder, the larger ones need fewer operand
// reads and widenings per product.  Row-major 4096 x 12288 (16 / 32 row tiles):
// 16 rows 31.6 / 78.5 us, 64 rows 100 / 107, 96 rows 143 / 156, 128 rows 182 /
// 160; 12288 x 4096: 96 rows 145 / 167, 128 rows 191 / 175.  (The 32-row
// natural-order tiles measured spill 30 and 40 registers: see k_project_tiles.)
constexpr uint64_t kTileFewRows = 96;

// vm_wait with no LDS operation outstanding either.
constexpr unsigned vm_lds_wait(unsigned n) { return 0x0070u | (n & 0xfu) | ((n >> 4) << 14); }

// A lane's operands of one tile for half a group (chain steps 4 half .. + 3):
// block b = lane / Edge, row lane % Edge.
template <class T, Order O>
struct Operands;

template <class T>
struct Operands<T, Order::kPermuted> {
  u32x2 v[T::W];  // four steps of chain kChains b + Split w + c
  __device__ __forceinline__ void load(const uint8_t* stage, int first_row, int half, int lane, int c) {
    const int b = lane / T::Edge, r = lane % T::Edge;
    const uint8_t* row = stage + (first_row + r) * T::kRowBytes + half / 2 * T::P * 16 + half % 2 * 8;
#pragma unroll
    for (int w = 0; w < T::W; ++w)
      v[w] = *reinterpret_cast<const u32x2*>(row + ((T::kChains * b + T::Split * w + c) ^ (r % 16)) * 16);
  }
  __device__ __forceinline__ float at(int w, int e, uint32_t) const {
    const uint32_t word = e < 2 ? v[w].x : v[w].y;
    return (e & 1) ? dl_bf16_hi(word) : dl_bf16_lo(word);
  }
};

template <class T>
struct Operands<T, Order::kNatural> {
  uint32_t v[4][T::W];  // per step, the word that holds the input (half c % 2 of it)
  __device__ __forceinline__ void load(const uint8_t* stage, int first_row, int half, int lane, int c) {
    const int b = lane / T::Edge, r = lane % T::Edge;
    const uint8_t* row = stage + (first_row + r) * T::kRowBytes;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
#pragma unroll
      for (int w = 0; w < T::W; ++w) {
        const int input = T::P * (4 * half + e) + T::kChains * b + T::Split * w;
        v[e][w] = *reinterpret_cast<const uint32_t*>(row + ((input / 8) ^ (r % 16)) * 16 + (input % 8 + c / 2 * 2) * 2);
      }
    }
  }
  // `select` moves half c % 2 of a word into the upper half of a register.
  __device__ __forceinline__ float at(int w, int e, uint32_t select) const {
    return __uint_as_float(__builtin_amdgcn_perm(0u, v[e][w], select));
  }
};

template <int Edge>
struct Products;
template <>
struct Products<32> {
  typedef f32x32 Sum;
  static __device__ __forceinline__ Sum step(float a, float b, Sum c) {
    return __builtin_amdgcn_mfma_f32_32x32x1f32(a, b, c, 0, 0, 0);
  }
};
template <>
struct Products<16> {
  typedef f32x16 Sum;
  static __device__ __forceinline__ Sum step(float a, float b, Sum c) {
    return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, c, 0, 0, 0);
  }
};

// The sums of one workgroup tile over `stages` stages.  a_src(row, piece) and
// b_src(row, piece) give the address of 16-byte piece `piece` (below P) of
// output row / input row of the tile in the first group of 8 steps; the same
// piece of the next group lies a_step / b_step bytes further.  Each piece
// lands in LDS at piece ^ (row % 16) of its row, so an operand read spreads
// over the banks while the loads of 4 lanes stay 64 contiguous bytes.
//
// Stages pass through a ring of LDS buffers by direct global-to-LDS loads.
// Ahead of a stage's last half group, one barrier finds the next stage in LDS
// and every wavefront past its reads of this one, whose buffer the stage
// kRing later then takes; the operands of each half group are read while the
// one before is multiplied.  Loads past the last stage repeat it so that
// every wait counts the same loads.  The buffers are separate LDS objects: the
// compiler then adds no waits of its own between the loads in flight and the
// operand reads.
//
// finish(output, row, sum) receives four consecutive outputs `output` .. + 3
// of tile row `row`.
template <class T, class ASrc, class BSrc, class Finish>
__device__ __forceinline__ void tile_sums(int stages, uint32_t a_step, uint32_t b_step, ASrc&& a_src, BSrc&& b_src,
                                          Finish&& finish) {
  constexpr int kTileGroups = T::Edge == 32 ? 4 : 1;  // groups of four outputs per lane
  constexpr int kExchange = T::Split > 1 ? T::kWaves * kTileGroups * 64 * sizeof(f32x4) : 16;
  __shared__ __align__(1024) uint8_t s0[T::kStageBytes > kExchange ? T::kStageBytes : kExchange], s1[T::kStageBytes],
      s2[T::kRing > 2 ? T::kStageBytes : 16], s3[T::kRing > 3 ? T::kStageBytes : 16];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int c = wave % T::Split, tile = wave / T::Split;
  const int a_row = T::Edge * (tile / T::TN), b_row = T::Edge * (tile % T::TN);
  const uint32_t select = c % 2 ? 0x03020c0cu : 0x01000c0cu;

  const uint8_t* src[T::kLoads];
  uint32_t step[T::kLoads];
#pragma unroll
  for (int j = 0; j < T::kLoads; ++j) {
    const int slot = (T::kWaves * j + wave) * 64 + lane;
    const int row = slot / T::kPieces, piece = (slot % T::kPieces) ^ (row % 16);
    // A 1 KiB unit lies wholly in the weights or in the rows.
    const bool weights = (T::kWaves * j + wave) * 64 / T::kPieces < T::kOutputs;
    const uint32_t group = weights ? a_step : b_step;
    src[j] = reinterpret_cast<const uint8_t*>(weights ? a_src(row, piece % T::P) : b_src(row - T::kOutputs, piece % T::P)) +
             piece / T::P * group;
    step[j] = T::kGroups * group;
  }
  auto issue = [&](int s, uint8_t* buffer) {
#pragma unroll
    for (int j = 0; j < T::kLoads; ++j)
      __builtin_amdgcn_global_load_lds((const global_ptr*)(src[j] + static_cast<uint64_t>(s) * step[j]),
                                       (lds_ptr*)(buffer + (T::kWaves * j + wave) * 1024), 16, 0, 0);
  };

  typename Products<T::Edge>::Sum acc[T::W];
#pragma unroll
  for (int w = 0; w < T::W; ++w)
#pragma unroll
    for (int r = 0; r < T::kRegs; ++r) acc[w][r] = 0.0f;

  struct Half {
    Operands<T, T::kWeights> a;
    Operands<T, T::kRowOrder> b;
  } f[2];
  auto load_half = [&](const uint8_t* buffer, int half) {
    f[half % 2].a.load(buffer, a_row, half, lane, c);
    f[half % 2].b.load(buffer, T::kOutputs + b_row, half, lane, c);
  };
  auto multiply = [&](int half) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int w = 0; w < T::W; ++w)
        acc[w] = Products<T::Edge>::step(f[half % 2].a.at(w, e, select), f[half % 2].b.at(w, e, select), acc[w]);
  };

  constexpr int kAhead = (T::kRing - 2) * T::kLoads;  // loads in flight past the next stage's
  issue(0, s0);
  issue(min(1, stages - 1), s1);
  if constexpr (T::kRing > 2) issue(min(2, stages - 1), s2);
  if constexpr (T::kRing > 3) issue(min(3, stages - 1), s3);
  __builtin_amdgcn_s_waitcnt(vm_wait(kAhead + T::kLoads));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  load_half(s0, 0);
  int s = 0;
  auto one = [&](uint8_t* current, const uint8_t* next) {
#pragma unroll
    for (int half = 0; half < 2 * T::kGroups; ++half) {
      if (half + 1 < 2 * T::kGroups) {
        load_half(current, half + 1);
      } else {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(vm_lds_wait(kAhead));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        load_half(next, 0);
        issue(min(s + T::kRing, stages - 1), current);
      }
      multiply(half);
    }
    __builtin_amdgcn_sched_barrier(0);
    ++s;
  };
  while (s + T::kRing <= stages) {
    one(s0, s1);
    one(s1, T::kRing > 2 ? s2 : s0);
    if constexpr (T::kRing > 2) one(s2, T::kRing > 3 ? s3 : s0);
    if constexpr (T::kRing > 3) one(s3, s0);
  }
  if (s < stages) one(s0, s1);
  if (T::kRing > 2 && s < stages) one(s1, s2);
  if (T::kRing > 3 && s < stages) one(s2, s3);
  __builtin_amdgcn_s_waitcnt(vm_lds_wait(0));  // no load outlives the ring

  // Registers of a block: row lane % Edge, outputs 4 (lane / Edge) + i (and
  // + 8 g of a 32-wide tile).  The offsets from P / 2 down to kChains merge
  // the blocks, the next ones instructions.
  f32x4 part[kTileGroups];
#pragma unroll
  for (int g = 0; g < kTileGroups; ++g) {
    f32x4 sum[T::W];
#pragma unroll
    for (int w = 0; w < T::W; ++w)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (T::Edge == 32)
          sum[w][i] = acc[w][4 * g + i] + acc[w][16 + 4 * g + i];
        else
          sum[w][i] = (acc[w][i] + acc[w][8 + i]) + (acc[w][4 + i] + acc[w][12 + i]);
      }
#pragma unroll
    for (int off = T::W / 2; off; off /= 2)
#pragma unroll
      for (int w = 0; w < off; ++w)
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[w][i] = sum[w][i] + sum[w + off][i];
    part[g] = sum[0];
  }
  if constexpr (T::Split == 1) {
#pragma unroll
    for (int g = 0; g < kTileGroups; ++g) finish(a_row + 8 * g + 4 * (lane / T::Edge), b_row + lane % T::Edge, part[g]);
    return;
  }
  // The remaining offsets across the tile's wavefronts through LDS.
  // Wavefront c finishes its share of the tile: whole groups while there are
  // enough, else a share of the lanes of one group.
  f32x4* exchange = reinterpret_cast<f32x4*>(s0);  // [tile][c][group][lane]
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int g = 0; g < kTileGroups; ++g) exchange[((tile * T::Split + c) * kTileGroups + g) * 64 + lane] = part[g];
  __syncthreads();
  constexpr int kShare = kTileGroups >= T::Split ? kTileGroups / T::Split : 1;  // groups per wavefront
  constexpr int kLanes = kTileGroups >= T::Split ? 1 : T::Split / kTileGroups;  // wavefronts per group
#pragma unroll
  for (int i = 0; i < kShare; ++i) {
    const int g = kLanes > 1 ? c / kLanes : c * kShare + i;
    if (kLanes > 1 && lane / (64 / kLanes) != c % kLanes) continue;
    f32x4 sum[T::Split];
#pragma unroll
    for (int k = 0; k < T::Split; ++k) sum[k] = exchange[((tile * T::Split + k) * kTileGroups + g) * 64 + lane];
#pragma unroll
    for (int off = T::Split / 2; off; off /= 2)
#pragma unroll
      for (int k = 0; k < off; ++k)
#pragma unroll
        for (int j = 0; j < 4; ++j) sum[k][j] = sum[k][j] + sum[k + off][j];
    finish(a_row + 8 * g + 4 * (lane / T::Edge), b_row + lane % T::Edge, sum[0]);
  }
}

}  // namespace dl::exact
