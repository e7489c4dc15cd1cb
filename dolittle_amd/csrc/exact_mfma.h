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

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x32 __attribute__((ext_vector_type(32)));
typedef __attribute__((address_space(3))) void lds_ptr;
typedef __attribute__((address_space(1))) void global_ptr;

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;

enum class Order { kPermuted, kNatural };

// A workgroup of 8 wavefronts computes TM x TN tiles of 32 outputs x 32 rows;
// Split wavefronts share a tile, each with P / Split of its chains (16 P /
// Split accumulators per lane).  Block b of instruction w of wavefront c holds
// chain t = (P / 2) b + Split w + c, so offsets P/2 .. Split merge inside a
// lane and only the last log2(Split) offsets cross wavefronts.
template <int P_, int Split_, int TM_, int TN_, int Ring_, Order Weights_>
struct Tile {
  static constexpr int P = P_, Split = Split_, TM = TM_, TN = TN_, kRing = Ring_;
  static constexpr Order kWeights = Weights_;
  static constexpr int W = P / Split / 2;  // instructions per chain step
  static constexpr int kOutputs = 32 * TM, kRows = 32 * TN;
  static constexpr int kStageRows = kOutputs + kRows;
  static constexpr int kRowBytes = 16 * P;  // 8 P inputs in BF16
  static constexpr int kInputs = 8 * P;     // inputs per stage
  static constexpr int kLoads = kStageRows * P / 64 / kWaves;  // 1 KiB loads per wavefront and stage
  static constexpr int kStageBytes = kStageRows * kRowBytes;
  static_assert(TM * TN * Split == kWaves && (P == 16 || P == 32), "eight wavefronts, 16 or 32 partials");
  static_assert(W == 2 || W == 4, "64 or 128 accumulators per lane");
  static_assert(kRing == 2 || kRing == 3, "two or three stage buffers");
};

// s_waitcnt immediates: at most n vector-memory operations outstanding (vmcnt
// bits 3:0 and 15:14; expcnt and lgkmcnt at their no-wait maxima); the same
// and no LDS operation outstanding.
constexpr unsigned vm_wait(unsigned n) { return 0x0f70u | (n & 0xfu) | ((n >> 4) << 14); }
constexpr unsigned vm_lds_wait(unsigned n) { return 0x0070u | (n & 0xfu) | ((n >> 4) << 14); }

// A lane's operands of one 32-row tile for half a stage (chain steps 4 half ..
// + 3): block b = lane / 32, row lane % 32.
template <class T, Order O>
struct Operands;

template <class T>
struct Operands<T, Order::kPermuted> {
  u32x2 v[T::W];  // four steps of chain (P / 2) b + Split w + c
  __device__ __forceinline__ void load(const uint8_t* stage, int first_row, int half, int lane, int c) {
    const int b = lane / 32, r = lane % 32;
    const uint8_t* row = stage + (first_row + r) * T::kRowBytes + half * 8;
#pragma unroll
    for (int w = 0; w < T::W; ++w)
      v[w] = *reinterpret_cast<const u32x2*>(row + ((T::P / 2 * b + T::Split * w + c) ^ (r % 16)) * 16);
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
    const int b = lane / 32, r = lane % 32;
    const uint8_t* row = stage + (first_row + r) * T::kRowBytes;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int base = T::P * (4 * half + e) + T::P / 2 * b;  // a multiple of 8
      if constexpr (T::Split == 2) {
        const u32x4 q = *reinterpret_cast<const u32x4*>(row + ((base / 8) ^ (r % 16)) * 16);
        v[e][0] = q.x;
        v[e][1] = q.y;
        v[e][2] = q.z;
        v[e][3] = q.w;
      } else {
#pragma unroll
        for (int w = 0; w < T::W; ++w) {
          const int input = base + T::Split * w;
          v[e][w] = *reinterpret_cast<const uint32_t*>(row + ((input / 8) ^ (r % 16)) * 16 + (input % 8) * 2 + c / 2 * 4);
        }
      }
    }
  }
  // `select` moves half c % 2 of a word into the upper half of a register.
  __device__ __forceinline__ float at(int w, int e, uint32_t select) const {
    return __uint_as_float(__builtin_amdgcn_perm(0u, v[e][w], select));
  }
};

// The sums of one workgroup tile over `stages` stages.  a_src(row, piece) and
// b_src(row, piece) give the address of a 16-byte piece of output row / input
// row of the tile in the first stage; the same piece of the next stage lies
// a_step / b_step bytes further.  Each piece lands in LDS at piece ^ (row % 16)
// of its row, so an operand read spreads over the banks while the loads of 4
// lanes stay 64 contiguous bytes.
//
// Stages pass through a ring of three LDS buffers by direct global-to-LDS
// loads.  Half way through a stage, one barrier finds the next stage in LDS
// and every wavefront past its reads of this one, whose buffer the stage
// after the next two then takes; the operands of each half are read while the
// half before is multiplied.  Loads past the last stage repeat it so that
// every wait counts the same loads.  The buffers are separate LDS objects: the
// compiler then adds no waits of its own between the loads in flight and the
// operand reads.
//
// finish(output, row, sum) receives four consecutive outputs `output` .. + 3
// of tile row `row`.
template <class T, class ASrc, class BSrc, class Finish>
__device__ __forceinline__ void tile_sums(int stages, uint32_t a_step, uint32_t b_step, ASrc&& a_src, BSrc&& b_src,
                                          Finish&& finish) {
  constexpr int kExchange = kWaves * 4 * 64 * sizeof(f32x4);
  __shared__ __align__(1024) uint8_t s0[T::kStageBytes > kExchange ? T::kStageBytes : kExchange], s1[T::kStageBytes],
      s2[T::kRing == 3 ? T::kStageBytes : 16];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int c = wave % T::Split, tile = wave / T::Split;
  const int a_row = 32 * (tile / T::TN), b_row = 32 * (tile % T::TN);
  const uint32_t select = c % 2 ? 0x03020c0cu : 0x01000c0cu;

  const uint8_t* src[T::kLoads];
  uint32_t step[T::kLoads];
#pragma unroll
  for (int j = 0; j < T::kLoads; ++j) {
    const int slot = (kWaves * j + wave) * 64 + lane;
    const int row = slot / T::P, piece = (slot % T::P) ^ (row % 16);
    // A 1 KiB unit lies wholly in the weights or in the rows.
    const bool weights = (kWaves * j + wave) * 64 / T::P < T::kOutputs;
    src[j] = reinterpret_cast<const uint8_t*>(weights ? a_src(row, piece) : b_src(row - T::kOutputs, piece));
    step[j] = weights ? a_step : b_step;
  }
  auto issue = [&](int s, uint8_t* buffer) {
#pragma unroll
    for (int j = 0; j < T::kLoads; ++j)
      __builtin_amdgcn_global_load_lds((const global_ptr*)(src[j] + static_cast<uint64_t>(s) * step[j]),
                                       (lds_ptr*)(buffer + (kWaves * j + wave) * 1024), 16, 0, 0);
  };

  f32x32 acc[T::W];
#pragma unroll
  for (int w = 0; w < T::W; ++w)
#pragma unroll
    for (int r = 0; r < 32; ++r) acc[w][r] = 0.0f;

  struct Half {
    Operands<T, T::kWeights> a;
    Operands<T, Order::kPermuted> b;
  };
  auto load_half = [&](const uint8_t* buffer, int half, Half& f) {
    f.a.load(buffer, a_row, half, lane, c);
    f.b.load(buffer, T::kOutputs + b_row, half, lane, c);
  };
  auto multiply = [&](const Half& f) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int w = 0; w < T::W; ++w)
        acc[w] = __builtin_amdgcn_mfma_f32_32x32x1f32(f.a.at(w, e, select), f.b.at(w, e, 0), acc[w], 0, 0, 0);
  };

  constexpr int kAhead = (T::kRing - 2) * T::kLoads;  // loads in flight past the next stage's
  issue(0, s0);
  issue(min(1, stages - 1), s1);
  if constexpr (T::kRing == 3) issue(min(2, stages - 1), s2);
  __builtin_amdgcn_s_waitcnt(vm_wait(kAhead + T::kLoads));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  Half f0, f1;
  load_half(s0, 0, f0);
  int s = 0;
  auto one = [&](uint8_t* current, const uint8_t* next) {
    load_half(current, 1, f1);
    multiply(f0);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(vm_lds_wait(kAhead));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    load_half(next, 0, f0);
    issue(min(s + T::kRing, stages - 1), current);
    multiply(f1);
    __builtin_amdgcn_sched_barrier(0);
    ++s;
  };
  if constexpr (T::kRing == 3) {
    while (s + 3 <= stages) {
      one(s0, s1);
      one(s1, s2);
      one(s2, s0);
    }
    if (s < stages) one(s0, s1);
    if (s < stages) one(s1, s2);
  } else {
    while (s + 2 <= stages) {
      one(s0, s1);
      one(s1, s0);
    }
    if (s < stages) one(s0, s1);
  }
  __builtin_amdgcn_s_waitcnt(vm_lds_wait(0));  // no load outlives the ring

  // Register r of a block: row lane % 32, output 8 (r / 4) + 4 (lane / 32) +
  // r % 4.  Offset P/2 merges the blocks, the next ones instructions.
  f32x4 part[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    f32x4 sum[T::W];
#pragma unroll
    for (int w = 0; w < T::W; ++w)
#pragma unroll
      for (int i = 0; i < 4; ++i) sum[w][i] = acc[w][4 * g + i] + acc[w][16 + 4 * g + i];
#pragma unroll
    for (int off = T::W / 2; off; off /= 2)
#pragma unroll
      for (int w = 0; w < off; ++w)
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[w][i] = sum[w][i] + sum[w + off][i];
    part[g] = sum[0];
  }
  // The remaining offsets across the tile's wavefronts through LDS: wavefront
  // c finishes the output groups [4 c / Split, 4 (c + 1) / Split); with eight
  // wavefronts per tile, the halves (lane / 32) of group c / 2.
  f32x4* exchange = reinterpret_cast<f32x4*>(s0);  // [tile][c][group][lane]
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int g = 0; g < 4; ++g) exchange[((tile * T::Split + c) * 4 + g) * 64 + lane] = part[g];
  __syncthreads();
  constexpr int kGroups = T::Split >= 4 ? 1 : 4 / T::Split;
#pragma unroll
  for (int i = 0; i < kGroups; ++i) {
    const int g = T::Split == 8 ? c / 2 : c * kGroups + i;
    if (T::Split == 8 && lane / 32 != c % 2) continue;
    f32x4 sum[T::Split];
#pragma unroll
    for (int k = 0; k < T::Split; ++k) sum[k] = exchange[((tile * T::Split + k) * 4 + g) * 64 + lane];
#pragma unroll
    for (int off = T::Split / 2; off; off /= 2)
#pragma unroll
      for (int k = 0; k < off; ++k)
#pragma unroll
        for (int j = 0; j < 4; ++j) sum[k][j] = sum[k][j] + sum[k + off][j];
    finish(a_row + 8 * g + 4 * (lane / 32), b_row + lane % 32, sum[0]);
  }
}

}  // namespace dl::exact
