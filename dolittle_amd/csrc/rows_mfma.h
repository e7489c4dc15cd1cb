// Packed exact-chain GEMVs of four or eight rows on depth-1 FP32 MFMA.
//
// v_mfma_f32_4x4x1_16b_f32 advances 16 chains of 4 outputs x 4 rows by one
// input each, one single-rounding FMA per element (bit-equal to fmaf, see
// exact_mfma.h): block b = lane / 4 is partial t, the lane's operand element
// output lane % 4 on one side and row lane % 4 on the other.  The packed
// weights (gemv.h) hold 8 consecutive elements of one chain in a 16-byte
// chunk, so a lane reads its chunk of the tile's 1 KiB step straight into
// registers, chunk (lane % 4) 16 + lane / 4 instead of chunk `lane`: the same
// contiguous kilobyte (a stream of such loads runs at 6.8-6.9 TB/s like one in
// lane order).
//
// Against one FMA per (row, element) on the vector ALUs with the inputs as FP32
// in LDS, a chunk of eight rows costs two 16-byte LDS reads instead of
// sixteen and the staged rows half the LDS (they are BF16 values).
//
// Staged rows.  Piece (g, c) is 1 KiB: chunk c of rows 4 g .. + 3, slot
// 4 t + (j ^ (t / 4)) holding the 8 elements of partial t of row 4 g + j, so
// that the reads of a wavefront and the 2-byte writes of 16 neighbouring
// inputs both spread over all banks.  P = 16: chunk c is step c; P = 32: chunk
// 2 s + h is step s of partials 16 h .. + 15.
#pragma once

#include "dl_device.h"
#include "gemv.h"

namespace dl::rows {

// 16-byte slot of partial t (below 16) of row j (below 4) in its piece.
__device__ __forceinline__ int slot_of(int t, int j) { return 4 * t + (j ^ (t / 4)); }

// BF16 element of input `col` of row `row` in the staged rows of `chunks`
// chunks (inputs / 128).
template <int P>
__device__ __forceinline__ int staged_element(int row, int col, int chunks) {
  const int t = col % P, m = col / P;
  const int c = m / 8 * (P / 16) + t / 16;
  return ((row / 4 * chunks + c) * 64 + slot_of(t % 16, row % 4)) * 8 + m % 8;
}

// Copies chunks [c0, c0 + N) of P-permuted rows (row stride `width` inputs) of
// R rows into `xs` by direct global-to-LDS loads; rows from `valid` on repeat
// the last one.
template <int R, int N, int Waves>
__device__ __forceinline__ void stage_permuted(const uint16_t* __restrict__ x, uint64_t width, int c0, int chunks,
                                               int valid, uint8_t* xs, int wave, int lane) {
  const int t = lane / 4, j = (lane % 4) ^ (t / 4);  // the slot's partial and row
  for (int piece = wave; piece < R / 4 * N; piece += Waves) {
    const int g = piece / N, c = c0 + piece % N;
    const uint16_t* src = x + static_cast<uint64_t>(min(4 * g + j, valid - 1)) * width +
                          (min(c, chunks - 1) * 16 + t) * 8;
    __builtin_amdgcn_global_load_lds((const global_ptr*)src, (lds_ptr*)(xs + piece * 1024), 16, 0, 0);
  }
}

__device__ __forceinline__ float element(u32x4 v, int e) {
  const uint32_t word = (e >> 1) == 0 ? v.x : (e >> 1) == 1 ? v.y : (e >> 1) == 2 ? v.z : v.w;
  return (e & 1) ? dl_bf16_hi(word) : dl_bf16_lo(word);
}

// One chunk: 8 inputs of 16 chains of 4 outputs for the G row groups; `x` is
// the lane's slot of the chunk's first piece, `group` slots between groups.
template <int G>
__device__ __forceinline__ void step(u32x4 w, const u32x4* x, int group, f32x4 (&acc)[G]) {
  u32x4 xv[G];
#pragma unroll
  for (int g = 0; g < G; ++g) xv[g] = x[g * group];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float a = element(w, e);
#pragma unroll
    for (int g = 0; g < G; ++g) acc[g] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, element(xv[g], e), acc[g], 0, 0, 0);
  }
}

// The lane's chunk offset in the 1 KiB step of a packed tile of four outputs
// (P = 16), or, with `half`, in the steps of the two packed tiles of four
// outputs (P = 32, partials 16 half .. + 15).
__device__ __forceinline__ uint64_t lane_chunk16(int lane) { return (lane % 4) * 16 + lane / 4; }
__device__ __forceinline__ uint64_t lane_chunk32(int lane, int half, int steps) {
  const int i = lane % 4;
  return static_cast<uint64_t>(i / 2) * steps * 64 + (i % 2) * 32 + 16 * half + lane / 4;
}

// `steps` chunks of one lane's chain (64 chunks apart from `src`), the staged
// piece of step s at x + s * stride.  Batches of kBatch chunks are
// double-buffered in registers; with `next`, its first batch is loaded during
// the last batch and left in `first`.  Needs an even number of whole batches
// for that; other counts go one chunk at a time.
template <int G>
__device__ __forceinline__ void chain(const u32x4* __restrict__ src, const u32x4* x, int stride, int group, int steps,
                                      f32x4 (&acc)[G], FirstBatch& first, const u32x4* __restrict__ next) {
  u32x4 wa[kBatch], wb[kBatch];
  auto load = [&](u32x4* w, const u32x4* from) {
#pragma unroll
    for (int j = 0; j < kBatch; ++j) w[j] = load_stream(from + j * 64);
  };
  if (steps % (2 * kBatch) != 0) {
    int s = 0;
    if (first.valid && steps >= kBatch) {
#pragma unroll
      for (int j = 0; j < kBatch; ++j) step<G>(first.w[j], x + j * stride, group, acc);
      s = kBatch;
    }
    for (; s < steps; ++s) step<G>(load_stream(src + s * 64), x + s * stride, group, acc);
    first.valid = false;
    return;
  }
  const bool has_next = __builtin_amdgcn_readfirstlane(next != nullptr ? 1 : 0) != 0;
  if (first.valid) {
#pragma unroll
    for (int j = 0; j < kBatch; ++j) wa[j] = first.w[j];
  } else {
    load(wa, src);
  }
  for (int s = 0; s < steps; s += 2 * kBatch) {
    load(wb, src + (s + kBatch) * 64);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < kBatch; ++j) step<G>(wa[j], x + (s + j) * stride, group, acc);
    __builtin_amdgcn_sched_barrier(0);
    // Past the last batch: the next chain's first, or this one again (still
    // in cache; a select, so both register sets stay in place).
    load(wa, s + 2 * kBatch < steps ? src + (s + 2 * kBatch) * 64 : (has_next ? next : src + (s + kBatch) * 64));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < kBatch; ++j) step<G>(wb[j], x + (s + kBatch + j) * stride, group, acc);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int j = 0; j < kBatch; ++j) first.w[j] = wa[j];
  first.valid = next != nullptr;
}

// Merges the 16 partials of every (output, row): offsets 8, 4, 2, 1 are lanes
// 32, 16, 8, 4 apart.  The first two exchange halves between two outputs, so
// both are added at once.  Returns, in lane 16 q + b (b < 4 G), the sum of row
// b for output output_of(q).
__device__ __forceinline__ int output_of(int q) { return (q & 1) * 2 + q / 2; }

template <int G>
__device__ __forceinline__ float merge(const f32x4 (&acc)[G], int lane) {
  auto halves = [](float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  };
  auto quarters = [](float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  };
  float n[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    n[g] = quarters(halves(acc[g][0], acc[g][1]), halves(acc[g][2], acc[g][3]));
    n[g] = n[g] + row_down<8>(n[g]);
    n[g] = n[g] + row_down<4>(n[g]);
  }
  if constexpr (G == 1) {
    return n[0];
  } else {
    // Rows 4 .. 7 move up four lanes (DPP row_shr:4).
    const float up = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(n[1]), 0x114, 0xf, 0xf, true));
    return lane % 16 < 4 ? n[0] : up;
  }
}

}  // namespace dl::rows
