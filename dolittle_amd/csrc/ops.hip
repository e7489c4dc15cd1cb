// The reference's eight-operation catalog on gfx950, operand layouts as the
// reference stores them (row-major W[O,I], Q[B,Hq,d], K/V[C,Hkv,d]).
//
// Each kernel restates one launch of src/kernels/cuda/launch.h:79-109 with
// the same reduction ownership, merge order and storage-rounding points, so
// results are bit-identical with the reference contract
// (docs/architecture/transformer-execution.md:115-170).  The wave64 mapping
// differs from the reference's warp32 mapping, but every reduction below is
// written so that the value produced is the reference tree's value:
//  - shuffle-down within a width-P segment returns the lane's own value when
//    the source lane leaves the segment, exactly like the CUDA intrinsic; the
//    lane that keeps the result therefore sees the identical pairing.
//  - exp, sin, cos, pow come from dl_math.h (deterministic, shared with the
//    CPU oracle); sqrt and division are IEEE correctly rounded.
#include <algorithm>
#include <cstdint>
#include <utility>
#include <type_traits>

#include "dl_device.h"
#include "dl_internal.h"
#include "exact_mfma.h"

namespace dl {
namespace {

constexpr int kThreads = 256;

inline unsigned grid_for(uint64_t tasks, uint64_t per_block, uint64_t cap = 1u << 30) {
  const uint64_t blocks = ceil_div(tasks, per_block);
  return static_cast<unsigned>(std::min<uint64_t>(std::max<uint64_t>(blocks, 1), cap));
}

// ----------------------------------------------------------------- projection
// projection.cu:277-318 (decode) and 218-275 (prefill): P lanes own one
// output; lane t is the FMA chain over features t, t+P, ...; a ragged input
// width emulates the tiled kernel's zero padding to 16 features
// (projection.cu:295-304); merge offsets P/2..1; round once.
template <class T, int P, int RT>
__global__ __launch_bounds__(kThreads) void projection_rowmajor(const T* __restrict__ x,
                                                                const T* __restrict__ w,
                                                                T* __restrict__ y, uint64_t rows,
                                                                uint64_t in_w, uint64_t out_w,
                                                                const uint64_t* out_pos) {
  constexpr int kOutputsPerBlock = kThreads / P;
  const int lane = threadIdx.x % P;
  const uint64_t o = static_cast<uint64_t>(blockIdx.x) * kOutputsPerBlock + threadIdx.x / P;
  const uint64_t r0 = static_cast<uint64_t>(blockIdx.y) * RT;
  const uint64_t base = out_pos ? *out_pos * out_w : 0;
  float acc[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) acc[r] = 0.0f;
  if (o < out_w) {
    const T* wr = w + o * in_w;
    for (uint64_t f = lane; f < in_w; f += P) {
      const float wv = load_elem(wr, f);
#pragma unroll
      for (int r = 0; r < RT; ++r)
        if (r0 + r < rows) acc[r] = fma_rn(load_elem(x + (r0 + r) * in_w, f), wv, acc[r]);
    }
    const uint64_t padded = ceil_div(in_w, 16) * 16;
    if (padded != in_w && static_cast<uint64_t>(lane) >= in_w % P &&
        static_cast<uint64_t>(lane) < (padded - 1) % P + 1) {
#pragma unroll
      for (int r = 0; r < RT; ++r) acc[r] = fma_rn(0.0f, 0.0f, acc[r]);
    }
  }
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    float v = acc[r];
#pragma unroll
    for (int off = P / 2; off; off >>= 1) v = v + __shfl_down(v, off, P);
    if (lane == 0 && o < out_w && r0 + r < rows) store_elem(y, base + (r0 + r) * out_w + o, v);
  }
}

// The same chains on the FP32 matrix cores (exact_mfma.h), row-major BF16
// operands in natural order: whole stages of inputs, 16-byte aligned rows.
// Rows and outputs past the end repeat the last one and are not stored.  Few
// rows are bound by the weight stream (16 rows of 4096 x 12288: 31 us, 3.2
// TB/s; 384 us with one lane per partial reading 2 bytes at a time), many by
// the FP32 MFMA rate and the operand widening.
//
// Wavefronts per SIMD, which bound the registers: the 32-row tiles (eight
// wavefronts, 64 and 80 KiB of LDS) are held at two workgroups per compute
// unit, 128 registers, and spill 30 (P = 16) and 40 (P = 32) of them to
// scratch inside the loop; the 16-row tiles take what their LDS leaves room
// for, two workgroups of four wavefronts (P = 16) or of eight (P = 32), and do
// not spill.
template <class T>
__global__ __launch_bounds__(T::kThreads) __attribute__((amdgpu_waves_per_eu(T::Edge == 32 ? 4 : T::P / 8)))
void k_project_tiles(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, uint16_t* __restrict__ y,
                     uint64_t rows, uint64_t in_w, uint64_t out_w, const uint64_t* out_pos) {
  const uint64_t id = blockIdx.x + static_cast<uint64_t>(blockIdx.y) * gridDim.x;
  // XCD x takes the output tiles x, x + 8, ..., all row tiles of one together.
  const bool by_xcd = gridDim.x % 8 == 0;
  const uint64_t tile = by_xcd ? id / 8 / gridDim.y * 8 + id % 8 : blockIdx.x;
  const uint64_t o0 = tile * T::kOutputs, r0 = (by_xcd ? id / 8 % gridDim.y : blockIdx.y) * T::kRows;
  uint16_t* out = y + (out_pos ? *out_pos * out_w : 0);
  const bool vector = out_w % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 8 == 0;
  exact::tile_sums<T>(
      static_cast<int>(in_w / T::kInputs), 16 * T::P, 16 * T::P,
      [&](int row, int piece) {
        return reinterpret_cast<const u32x4*>(w + min(o0 + row, out_w - 1) * in_w) + piece;
      },
      [&](int row, int piece) {
        return reinterpret_cast<const u32x4*>(x + min(r0 + row, rows - 1) * in_w) + piece;
      },
      [&](int output, int row, f32x4 sum) {
        const uint64_t r = r0 + row, o = o0 + output;
        if (r >= rows || o >= out_w) return;
        uint16_t v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = dl_f32_to_bf16(sum[i]);
        uint16_t* at = out + r * out_w + o;
        if (vector) {
          *reinterpret_cast<u32x2*>(at) = u32x2{v[0] | (static_cast<uint32_t>(v[1]) << 16),
                                                v[2] | (static_cast<uint32_t>(v[3]) << 16)};
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (o + i < out_w) at[i] = v[i];
        }
      });
}

// One row, bound by the weight stream.  A wavefront owns 8 outputs, 8 lanes
// each: lane (r, j) holds the P / 8 chains (P / 8) j .. of output r, which are
// neighbours in a row-major row, so one LDS read brings a step of all of them.
// Its weights stream through its own ring of kRing LDS buffers (256 inputs of
// 8 rows, 4 KiB) by direct global-to-LDS loads, so what is in flight takes no
// registers and no wavefront waits for another; the input row is staged once
// per workgroup as FP32.  Piece p of row r lies at p ^ (P / 8 r): the 8 rows of
// a read fall in distinct banks.
//
// Measured (one lane per partial reading 2 bytes at a time / the matrix-core
// tiles of 16 rows / this): 4096 x 4096 98 / 14.5 / 12.4 us, 4096 x 1024 59 /
// 13 / 9.7, 4096 x 12288 166 / 31 / 22.3 (4.5 TB/s), 12288 x 4096 185 / 34 /
// 29, 4096 x 151936 202 us (6.2 TB/s).
template <int P_, int MaxInputs_>
struct RowTile {
  static constexpr int P = P_, kMaxInputs = MaxInputs_, kWaves = 2, kRing = 4;
  static constexpr int kRows = 8, C = P / 8;  // outputs per wavefront, chains per lane
  static constexpr int kInputs = 256, kRowBytes = 2 * kInputs, kPieces = kInputs / 8;
  static constexpr int kStageBytes = kRows * kRowBytes, kLoads = kStageBytes / 1024;
  static constexpr int kThreads = 64 * kWaves;
};

template <int... I, class F>
__device__ __forceinline__ void for_each_index(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}

// Stage buffer I of every wavefront: a separate LDS object per stage, so the
// compiler adds no waits between the loads in flight and the reads.
template <class T, int I>
__device__ __forceinline__ uint8_t* row_stage(int wave) {
  __shared__ __align__(1024) uint8_t stage[T::kWaves * T::kStageBytes];
  return stage + wave * T::kStageBytes;
}

template <class T>
__global__ __launch_bounds__(T::kThreads) void k_project_row(const uint16_t* __restrict__ x,
                                                             const uint16_t* __restrict__ w, uint16_t* __restrict__ y,
                                                             uint64_t in_w, uint64_t out_w, const uint64_t* out_pos) {
  constexpr int P = T::P, C = T::C;
  // Static: reads of dynamic LDS would wait for every load in flight.
  __shared__ __align__(16) float xs[T::kMaxInputs];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int r = lane / 8, j = lane % 8;
  const uint64_t o0 = (static_cast<uint64_t>(blockIdx.x) * T::kWaves + wave) * T::kRows;
  const int stages = static_cast<int>(in_w / T::kInputs), chunks = static_cast<int>(in_w / 8);

  // The input comes before the weights: loads retire in order.
  constexpr int kChunks = T::kMaxInputs / 8 / T::kThreads;
  u32x4 xv[kChunks];
#pragma unroll
  for (int i = 0; i < kChunks; ++i)
    xv[i] = reinterpret_cast<const u32x4*>(x)[min(static_cast<int>(threadIdx.x) + i * T::kThreads, chunks - 1)];
  __builtin_amdgcn_sched_barrier(0);
  const uint8_t* src[T::kLoads];
#pragma unroll
  for (int i = 0; i < T::kLoads; ++i) {
    const int slot = i * 64 + lane, row = slot / T::kPieces, piece = (slot % T::kPieces) ^ (C * row % T::kPieces);
    src[i] = reinterpret_cast<const uint8_t*>(w + min(o0 + row, out_w - 1) * in_w) + piece * 16;
  }
  auto issue = [&](int s, uint8_t* buffer) {
#pragma unroll
    for (int i = 0; i < T::kLoads; ++i)
      __builtin_amdgcn_global_load_lds((const global_ptr*)(src[i] + static_cast<uint64_t>(s) * T::kRowBytes),
                                       (lds_ptr*)(buffer + i * 1024), 16, 0, 0);
  };
  for_each_index(std::make_integer_sequence<int, T::kRing>{}, [&](auto i) {
    issue(min(static_cast<int>(i.value), stages - 1), row_stage<T, i.value>(wave));
  });
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < kChunks; ++i) {
    const int chunk = threadIdx.x + i * T::kThreads;
    if (chunk < chunks) {
      float4* dst = reinterpret_cast<float4*>(xs + 8 * chunk);
      dst[0] = make_float4(dl_bf16_lo(xv[i].x), dl_bf16_hi(xv[i].x), dl_bf16_lo(xv[i].y), dl_bf16_hi(xv[i].y));
      dst[1] = make_float4(dl_bf16_lo(xv[i].z), dl_bf16_hi(xv[i].z), dl_bf16_lo(xv[i].w), dl_bf16_hi(xv[i].w));
    }
  }
  __syncthreads();

  float acc[C];
#pragma unroll
  for (int i = 0; i < C; ++i) acc[i] = 0.0f;
  auto one = [&](int s, uint8_t* buffer) {
    __builtin_amdgcn_s_waitcnt(vm_wait((T::kRing - 1) * T::kLoads));  // stage s has landed
    __builtin_amdgcn_sched_barrier(0);
    const uint8_t* row = buffer + r * T::kRowBytes;
    const float* xt = xs + s * T::kInputs + C * j;
    const int swizzle = C * r % T::kPieces;
#pragma unroll
    for (int e = 0; e < T::kInputs / P; ++e) {
      const int input = P * e + C * j;
      const uint8_t* at = row + ((input / 8) ^ swizzle) * 16 + (input % 8) * 2;
      if constexpr (C == 2) {
        const uint32_t v = *reinterpret_cast<const uint32_t*>(at);
        const float2 xe = *reinterpret_cast<const float2*>(xt + P * e);
        acc[0] = fma_rn(xe.x, dl_bf16_lo(v), acc[0]);
        acc[1] = fma_rn(xe.y, dl_bf16_hi(v), acc[1]);
      } else {
        const u32x2 v = *reinterpret_cast<const u32x2*>(at);
        const float4 xe = *reinterpret_cast<const float4*>(xt + P * e);
        acc[0] = fma_rn(xe.x, dl_bf16_lo(v.x), acc[0]);
        acc[1] = fma_rn(xe.y, dl_bf16_hi(v.x), acc[1]);
        acc[2] = fma_rn(xe.z, dl_bf16_lo(v.y), acc[2]);
        acc[3] = fma_rn(xe.w, dl_bf16_hi(v.y), acc[3]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xc07f);  // the buffer is read: stage s + kRing may take it
    issue(min(s + T::kRing, stages - 1), buffer);
  };
  for (int s = 0; s < stages; s += T::kRing) {
    for_each_index(std::make_integer_sequence<int, T::kRing>{}, [&](auto i) {
      if (s + i.value < stages) one(s + i.value, row_stage<T, i.value>(wave));
    });
  }
  __builtin_amdgcn_s_waitcnt(vm_wait(0));  // no load outlives the wavefront

  // Offsets P / 2 .. C across the output's lanes, the rest within the lane.
#pragma unroll
  for (int i = 0; i < C; ++i) {
    acc[i] = acc[i] + row_down<4>(acc[i]);
    acc[i] = acc[i] + row_down<2>(acc[i]);
    acc[i] = acc[i] + row_down<1>(acc[i]);
  }
#pragma unroll
  for (int off = C / 2; off; off /= 2)
#pragma unroll
    for (int i = 0; i < off; ++i) acc[i] = acc[i] + acc[i + off];
  if (j == 0 && o0 + r < out_w) y[(out_pos ? *out_pos * out_w : 0) + o0 + r] = dl_f32_to_bf16(acc[0]);
}

template <class T>
void launch_project_row(hipStream_t s, const uint16_t* x, const uint16_t* w, uint16_t* y, uint64_t in_w,
                        uint64_t out_w, const uint64_t* out_pos) {
  k_project_row<T><<<static_cast<unsigned>(ceil_div(out_w, T::kRows * T::kWaves)), T::kThreads, 0, s>>>(
      x, w, y, in_w, out_w, out_pos);
}

// Whether a BF16 projection runs on k_project_tiles: whole stages of 256
// inputs and 16-byte aligned operands.
bool tiled_projection(const void* x, const void* w, uint64_t in_w) {
  return in_w % 256 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0;
}

void launch_project_tiles(hipStream_t s, const uint16_t* x, const uint16_t* w, uint16_t* y, uint64_t rows,
                          uint64_t in_w, uint64_t out_w, const uint64_t* out_pos) {
  using namespace exact;
  constexpr Order kN = Order::kNatural;
  auto run = [&](auto tile) {
    using T = decltype(tile);
    const dim3 grid(static_cast<unsigned>(ceil_div(out_w, T::kOutputs)), static_cast<unsigned>(ceil_div(rows, T::kRows)));
    k_project_tiles<T><<<grid, T::kThreads, 0, s>>>(x, w, y, rows, in_w, out_w, out_pos);
  };
  if (rows == 1 && in_w <= 12288) {  // the input row as FP32 in LDS
    if (in_w <= 4096 && out_w > 1024)
      launch_project_row<RowTile<16, 4096>>(s, x, w, y, in_w, out_w, out_pos);
    else if (in_w <= 4096)
      launch_project_row<RowTile<32, 4096>>(s, x, w, y, in_w, out_w, out_pos);
    else
      launch_project_row<RowTile<32, 12288>>(s, x, w, y, in_w, out_w, out_pos);
    return;
  }
  if (in_w <= 4096 && out_w > 1024) {
    if (rows <= kTileFewRows)
      run(Tile<16, 16, 4, 1, 1, 2, 4, kN, kN>{});
    else
      run(Tile<16, 32, 4, 2, 1, 1, 3, kN, kN>{});
  } else {
    if (rows <= kTileFewRows)
      run(Tile<32, 16, 8, 1, 1, 1, 4, kN, kN>{});
    else
      run(Tile<32, 32, 8, 1, 1, 1, 2, kN, kN>{});
  }
}

template <class T>
void launch_projection_rowmajor(hipStream_t s, const void* x, const void* w, void* y, uint64_t rows,
                                uint64_t in_w, uint64_t out_w, const uint64_t* out_pos) {
  constexpr int RT = 8;
  const bool narrow = in_w <= 4096 && out_w > 1024;
  const uint64_t row_blocks = ceil_div(rows, RT);
  require(row_blocks <= 65535, "projection rows exceed the launch limit", DL_LENGTH_ERROR);
  if constexpr (std::is_same_v<T, uint16_t>) {
    if (tiled_projection(x, w, in_w)) {
      launch_project_tiles(s, static_cast<const T*>(x), static_cast<const T*>(w), static_cast<T*>(y), rows, in_w, out_w,
                           out_pos);
      return;
    }
  }
  if (narrow) {
    dim3 grid(grid_for(out_w, kThreads / 16), static_cast<unsigned>(row_blocks));
    projection_rowmajor<T, 16, RT><<<grid, kThreads, 0, s>>>(
        static_cast<const T*>(x), static_cast<const T*>(w), static_cast<T*>(y), rows, in_w, out_w, out_pos);
  } else {
    dim3 grid(grid_for(out_w, kThreads / 32), static_cast<unsigned>(row_blocks));
    projection_rowmajor<T, 32, RT><<<grid, kThreads, 0, s>>>(
        static_cast<const T*>(x), static_cast<const T*>(w), static_cast<T*>(y), rows, in_w, out_w, out_pos);
  }
}

// ------------------------------------------------------------------ rms norm
// normalization.cu:82-186.  Thread i < 128 is lane t = i/4, component c = i%4:
// width > 128 sums squares of features 4t+c+128k; width <= 128 holds feature
// t+32c.  Components combine left to right, lanes reduce with shuffle-down
// offsets 1..16, inverse = 1/sqrt(total * FP32(1/width) + eps),
// y = round(round(x * inverse) * w).
//
// Wide: eight loads in flight per thread, the squares still added in ascending
// order, from the width at which a thread has eight values (1 row of 4096 BF16
// 7.8 -> 5.3 us, 40,000 of 1000 92 -> 69).  Below it the check for a whole batch
// only costs: 40,000 rows of 192 or 256 take 31.0 and 33.4 us without it, 32.0
// and 35.0 with it.
constexpr uint64_t kWideNorm = 7 * 128 + 1;

template <class T, bool Wide>
__global__ __launch_bounds__(kThreads) void rms_norm_rows(const T* __restrict__ x,
                                                          const T* __restrict__ w,
                                                          T* __restrict__ y, uint64_t rows,
                                                          uint64_t width, float eps) {
  __shared__ float lanes[32];
  __shared__ float inverse_shared;
  for (uint64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    const T* xr = x + row * width;
    if (threadIdx.x < 128) {
      const unsigned t = threadIdx.x / 4, c = threadIdx.x % 4;
      float comp = 0.0f;
      if (width <= 128) {
        const uint64_t col = t + 32u * c;
        if (col < width) {
          const float v = load_elem(xr, col);
          comp = v * v;
        }
      } else {
        uint64_t col = 4u * t + c;
        if constexpr (Wide) {
          for (; col + 7 * 128 < width; col += 8 * 128) {
            float v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = load_elem(xr, col + 128 * k);
#pragma unroll
            for (int k = 0; k < 8; ++k) comp = comp + v[k] * v[k];
          }
        }
        for (; col < width; col += 128) {
          const float v = load_elem(xr, col);
          comp = comp + v * v;
        }
      }
      const float second = __shfl_down(comp, 1, 4);
      const float third = __shfl_down(comp, 2, 4);
      const float fourth = __shfl_down(comp, 3, 4);
      if (c == 0) lanes[t] = ((comp + second) + third) + fourth;
    }
    __syncthreads();
    if (threadIdx.x < 32) {
      float s = lanes[threadIdx.x];
#pragma unroll
      for (int off = 1; off < 32; off *= 2) s = s + __shfl_down(s, off, 32);
      if (threadIdx.x == 0) inverse_shared = inverse_sqrt(s * (1.0f / static_cast<float>(width)) + eps);
    }
    __syncthreads();
    const float inverse = inverse_shared;
    for (uint64_t col = threadIdx.x; col < width; col += blockDim.x) {
      const float normalized = storage_round<T>(load_elem(xr, col) * inverse);
      store_elem(y, row * width + col, normalized * load_elem(w, col));
    }
    __syncthreads();
  }
}

// -------------------------------------------------------------------- rotary
// rotary.cu:84-126.
template <class T>
__global__ __launch_bounds__(kThreads) void rotary_pairs(const T* __restrict__ x, T* __restrict__ y,
                                                         uint64_t pairs, uint64_t heads,
                                                         uint64_t width, uint64_t host_first,
                                                         double theta, const uint64_t* dev_pos,
                                                         int positioned) {
  const uint64_t first = position_or(dev_pos, host_first);
  T* out = y + (positioned ? first * heads * width : 0);
  const uint64_t half = width / 2;
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t idx = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; idx < pairs;
       idx += stride) {
    const uint64_t feature = idx % half, row = idx / half;
    const uint64_t position = first + row / heads;
    const float exponent = static_cast<float>(2 * feature) / static_cast<float>(width);
    const float inverse_frequency = static_cast<float>(1.0 / dl_pow_pos(theta, static_cast<double>(exponent)));
    const float angle = static_cast<float>(position) * inverse_frequency;
    double s, c;
    dl_sincos(static_cast<double>(angle), &s, &c);
    const float cosine = storage_round<T>(static_cast<float>(c));
    const float sine = storage_round<T>(static_cast<float>(s));
    const float a = load_elem(x, row * width + feature);
    const float b = load_elem(x, row * width + feature + half);
    const float ac = storage_round<T>(a * cosine), bs = storage_round<T>(b * sine);
    const float bc = storage_round<T>(b * cosine), as = storage_round<T>(a * sine);
    store_elem(out, row * width + feature, ac - bs);
    store_elem(out, row * width + feature + half, bc + as);
  }
}

// ----------------------------------------------------------------- attention
// attention.cu:231-383 (retained scores) and 436-439 (scale).
__global__ void attention_scale_kernel(float* out, uint64_t width) {
  *out = static_cast<float>(1.0 / __builtin_sqrt(static_cast<double>(width)));
}

template <class T>
__global__ __launch_bounds__(kThreads) void attention_retained(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, T* __restrict__ out,
    uint64_t tasks, uint64_t q_heads, uint64_t kv_heads, uint64_t width, uint64_t host_first,
    const float* scale_ptr, const uint64_t* dev_pos) {
  extern __shared__ float shared[];
  float* qs = shared;
  float* scores = qs + width;
  __shared__ float reduction[kThreads];
  __shared__ float denominator_shared;
  const unsigned tid = threadIdx.x;
  const unsigned lane = tid % 8, group = tid / 8;
  const uint64_t span = width / 8 + (width % 8 != 0);
  const float scale = *scale_ptr;
  for (uint64_t task = blockIdx.x; task < tasks; task += gridDim.x) {
    const uint64_t first = position_or(dev_pos, host_first);
    const uint64_t count = first + task / q_heads + 1;
    const uint64_t kvh = (task % q_heads) / (q_heads / kv_heads);
    for (uint64_t f = tid; f < width; f += blockDim.x) qs[f] = load_elem(q, task * width + f);
    __syncthreads();
    for (uint64_t base = 0; base < count; base += kThreads / 8) {
      const uint64_t j = base + group;
      float partial = 0.0f;
      if (j < count) {
        const uint64_t kv_offset = (j * kv_heads + kvh) * width;
        const uint64_t begin = lane * span;
        const uint64_t end = begin < width ? (begin + span < width ? begin + span : width) : width;
        for (uint64_t f = begin; f < end; ++f) partial = fma_rn(qs[f], load_elem(k, kv_offset + f), partial);
      }
#pragma unroll
      for (int off = 4; off; off >>= 1) partial = partial + __shfl_down(partial, off, 8);
      if (lane == 0 && j < count) scores[j] = partial * scale;
    }
    __syncthreads();
    float maximum = scores[0];
    for (uint64_t j = tid; j < count; j += blockDim.x) maximum = fmaxf(maximum, scores[j]);
    reduction[tid] = maximum;
    __syncthreads();
    for (unsigned off = kThreads / 2; off; off >>= 1) {
      if (tid < off) reduction[tid] = fmaxf(reduction[tid], reduction[tid + off]);
      __syncthreads();
    }
    maximum = reduction[0];
    __syncthreads();
    if (tid < 32) {
      float partial = 0.0f;
      for (uint64_t j = tid; j < count; j += 32) {
        const float e = dl_expf(scores[j] - maximum);
        scores[j] = e;
        partial = partial + e;
      }
#pragma unroll
      for (int off = 16; off; off >>= 1) partial = partial + __shfl_down(partial, off, 32);
      if (tid == 0) denominator_shared = partial;
    }
    __syncthreads();
    const float denominator = denominator_shared;
    for (uint64_t j = tid; j < count; j += blockDim.x) scores[j] = scores[j] / denominator;
    __syncthreads();
    const uint64_t split = (count - 1) / 2 + 1;
    if (width <= kThreads / 2) {
      const unsigned feature = tid % (kThreads / 2), half = tid / (kThreads / 2);
      const uint64_t begin = half == 0 ? 0 : split, end = half == 0 ? split : count;
      float sum = 0.0f;
      if (feature < width) {
        for (uint64_t j = begin; j < end; ++j)
          sum = fma_rn(scores[j], load_elem(v, (j * kv_heads + kvh) * width + feature), sum);
      }
      reduction[tid] = sum;
      __syncthreads();
      if (tid < width) store_elem(out, task * width + tid, reduction[tid] + reduction[tid + kThreads / 2]);
    } else {
      for (uint64_t feature = tid; feature < width; feature += blockDim.x) {
        float a = 0.0f, b = 0.0f;
        for (uint64_t j = 0; j < split; ++j)
          a = fma_rn(scores[j], load_elem(v, (j * kv_heads + kvh) * width + feature), a);
        for (uint64_t j = split; j < count; ++j)
          b = fma_rn(scores[j], load_elem(v, (j * kv_heads + kvh) * width + feature), b);
        store_elem(out, task * width + feature, a + b);
      }
    }
    __syncthreads();
  }
}

// 16 consecutive features in FP32; 16-byte aligned.
__device__ __forceinline__ void load_features(const uint16_t* p, float (&v)[16]) {
  const u32x4* q = reinterpret_cast<const u32x4*>(p);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const u32x4 w = q[i];
    v[8 * i + 0] = dl_bf16_lo(w.x); v[8 * i + 1] = dl_bf16_hi(w.x);
    v[8 * i + 2] = dl_bf16_lo(w.y); v[8 * i + 3] = dl_bf16_hi(w.y);
    v[8 * i + 4] = dl_bf16_lo(w.z); v[8 * i + 5] = dl_bf16_hi(w.z);
    v[8 * i + 6] = dl_bf16_lo(w.w); v[8 * i + 7] = dl_bf16_hi(w.w);
  }
}
__device__ __forceinline__ void load_features(const float* p, float (&v)[16]) {
  const float4* q = reinterpret_cast<const float4*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float4 w = q[i];
    v[4 * i] = w.x; v[4 * i + 1] = w.y; v[4 * i + 2] = w.z; v[4 * i + 3] = w.w;
  }
}

// attention_retained for heads of 128 features on 16-byte aligned rows: the
// same ranges, merges and rounding points (attention.cu:231-383) with the
// latencies overlapped.  Every thread keeps several key rows in flight, all
// threads take part in the exponentials, and the two PV chains of a feature
// read 16 keys ahead.  One workgroup per (position, query head), numbered so
// that the heads of a K/V group run on one XCD.  Bound: at one row the issue
// of the chains' instructions (load, widening, FMA per key); 16 rows at 1024
// keys 321 -> 43 us, one row at 512 keys 138 -> 24 us, at 4000 keys 107 us.
constexpr int kRowThreads = 512;
constexpr int kHeadWidth = 128;

template <class T>
__global__ __launch_bounds__(kRowThreads) void attention_heads(const T* __restrict__ q, const T* __restrict__ k,
                                                               const T* __restrict__ v, T* __restrict__ out,
                                                               uint64_t tasks, uint32_t q_heads, uint32_t kv_heads,
                                                               uint64_t host_first, const float* scale_ptr,
                                                               const uint64_t* dev_pos) {
  extern __shared__ __align__(16) float scores[];
  __shared__ float wave_values[kRowThreads / 64];
  __shared__ float denominator_shared;
  __shared__ float halves[2 * kHeadWidth];
  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int part = tid % 8, group = tid / 8;  // 8 lanes per key, 16 features each
  const uint32_t ratio = q_heads / kv_heads;
  const uint64_t stride = static_cast<uint64_t>(kv_heads) * kHeadWidth;
  const float scale = *scale_ptr;
  const uint64_t first = position_or(dev_pos, host_first);
  for (uint64_t id = blockIdx.x; id < tasks; id += gridDim.x) {
    const uint32_t in_row = static_cast<uint32_t>(id % q_heads);
    const uint32_t kvh = in_row % kv_heads;
    const uint64_t task = id - in_row + kvh * ratio + in_row / kv_heads;
    const int count = static_cast<int>(first + id / q_heads + 1);
    const T* krow = k + static_cast<uint64_t>(kvh) * kHeadWidth + 16 * part;
    float qv[16];
    load_features(q + task * kHeadWidth + 16 * part, qv);
    constexpr int kKeys = kRowThreads / 8, kAhead = sizeof(T) == 2 ? 4 : 2;
    float maximum = -INFINITY;
    // Scores of N passes of 64 keys from `base` on, all their key rows in
    // flight, and the maximum over the thread's own; a NaN score is ignored, as
    // fmaxf does in any order.  `whole`: every key of the passes is visible.
    auto pass = [&](auto n, auto whole, int base) {
      constexpr int N = decltype(n)::value;
      constexpr bool kWhole = decltype(whole)::value;
      float kv[N][16];
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int j = base + i * kKeys + group;
        load_features(krow + static_cast<uint64_t>(kWhole ? j : min(j, count - 1)) * stride, kv[i]);
      }
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int j = base + i * kKeys + group;
        float partial = 0.0f;
#pragma unroll
        for (int f = 0; f < 16; ++f) partial = fma_rn(qv[f], kv[i][f], partial);
        partial = partial + row_down<4>(partial);
        partial = partial + row_down<2>(partial);
        partial = partial + row_down<1>(partial);
        if (part == 0 && (kWhole || j < count)) {
          const float s = partial * scale;
          scores[j] = s;
          maximum = fmaxf(maximum, s);
        }
      }
    };
    // A wavefront takes no more passes than it has keys for: rows at short
    // positions leave most slots of kAhead passes empty.  FP32 rows keep half
    // as many in flight, the bytes of four BF16 ones: 109 registers, so two
    // workgroups per compute unit (143 and one with four).  FP32, 32 heads,
    // against four clamped passes throughout: 64 rows from position 0 43 -> 20
    // us (the general kernel 27), 16 rows at 1024 keys 52 -> 39, one row at 8000
    // 174 -> 170; BF16 within 2%, 64 rows from position 0 20 -> 17.5 us.
    int base = 0;
    for (; base + kAhead * kKeys <= count; base += kAhead * kKeys)
      pass(std::integral_constant<int, kAhead>{}, std::true_type{}, base);
    const int left = count - base - 8 * wave;  // keys from the wavefront's first on
    if (kAhead > 2 && left > 2 * kKeys)
      pass(std::integral_constant<int, kAhead>{}, std::false_type{}, base);
    else if (left > kKeys)
      pass(std::integral_constant<int, 2>{}, std::false_type{}, base);
    else if (left > 0)
      pass(std::integral_constant<int, 1>{}, std::false_type{}, base);
    maximum = wave_max(maximum);
    if (lane == 0) wave_values[wave] = maximum;
    __syncthreads();
    // NaN scores are ignored; if all are NaN the maximum is -infinity where the
    // reference's is NaN, and the differences below are NaN either way.
#pragma unroll
    for (int w = 0; w < kRowThreads / 64; ++w) maximum = fmaxf(maximum, wave_values[w]);
    for (int j = tid; j < count; j += kRowThreads) scores[j] = dl_expf(scores[j] - maximum);
    __syncthreads();
    if (tid < 32) {
      float partial = 0.0f;
      int j = tid;
      for (; j + 15 * 32 < count; j += 16 * 32) {
        float e[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) e[i] = scores[j + 32 * i];
#pragma unroll
        for (int i = 0; i < 16; ++i) partial = partial + e[i];
      }
      for (; j < count; j += 32) partial = partial + scores[j];
#pragma unroll
      for (int off = 16; off; off >>= 1) partial = partial + __shfl_down(partial, off, 32);
      if (tid == 0) denominator_shared = partial;
    }
    __syncthreads();
    const float denominator = denominator_shared;
    for (int j = tid; j < count; j += kRowThreads) scores[j] = scores[j] / denominator;
    __syncthreads();
    if (tid < 2 * kHeadWidth) {
      const int split = (count - 1) / 2 + 1, feature = tid % kHeadWidth, half = tid / kHeadWidth;
      const int end = half ? count : split;
      const T* vrow = v + static_cast<uint64_t>(kvh) * kHeadWidth + feature;
      float sum = 0.0f;
      int j = half ? split : 0;
      for (; j < end && j % 4; ++j) sum = fma_rn(scores[j], load_elem(vrow, j * stride), sum);
      constexpr int kBatch = 16;
      T va[kBatch], vb[kBatch];
      auto load = [&](T (&x)[kBatch], int at) {  // past the range: its last key again
#pragma unroll
        for (int i = 0; i < kBatch; ++i) x[i] = vrow[static_cast<uint64_t>(min(at + i, end - 1)) * stride];
      };
      auto chain = [&](const T (&x)[kBatch], int at) {
#pragma unroll
        for (int i = 0; i < kBatch; i += 4) {
          const float4 p = *reinterpret_cast<const float4*>(scores + at + i);
          sum = fma_rn(p.x, load_elem(x, i), sum);
          sum = fma_rn(p.y, load_elem(x, i + 1), sum);
          sum = fma_rn(p.z, load_elem(x, i + 2), sum);
          sum = fma_rn(p.w, load_elem(x, i + 3), sum);
        }
      };
      const int batches = (end - j) / kBatch;
      if (batches > 0) load(va, j);
      for (int b = 0; b < batches; b += 2) {
        load(vb, j + kBatch);
        chain(va, j);
        j += kBatch;
        if (b + 1 < batches) {
          load(va, j + kBatch);
          chain(vb, j);
          j += kBatch;
        }
      }
      for (; j < end; ++j) sum = fma_rn(scores[j], load_elem(vrow, j * stride), sum);
      halves[tid] = sum;
    }
    __syncthreads();
    if (tid < kHeadWidth) store_elem(out, task * kHeadWidth + tid, halves[tid] + halves[tid + kHeadWidth]);
    __syncthreads();
  }
}

// -------------------------------------------------------- embedding, add, silu
// embedding.cu:60-80; a token outside the table writes zeros instead of
// reading out of bounds.
template <class Bits>
__global__ __launch_bounds__(kThreads) void embedding_rows(const uint32_t* __restrict__ tokens,
                                                           const Bits* __restrict__ table,
                                                           Bits* __restrict__ out, uint64_t rows,
                                                           uint64_t width, uint64_t vocabulary) {
  for (uint64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    const uint32_t token = tokens[row];
    for (uint64_t f = threadIdx.x; f < width; f += blockDim.x)
      out[row * width + f] = token < vocabulary ? table[static_cast<uint64_t>(token) * width + f] : Bits(0);
  }
}

// elementwise.cu:2-18, 62-87.
template <class T, bool Silu>
__global__ __launch_bounds__(kThreads) void elementwise(const T* __restrict__ left,
                                                        const T* __restrict__ right,
                                                        T* __restrict__ out, uint64_t count) {
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += stride) {
    const float a = load_elem(left, i), b = load_elem(right, i);
    float result;
    if constexpr (Silu) {
      const float e = dl_expf(a >= 0.0f ? -a : a);
      const float sigmoid = a >= 0.0f ? 1.0f / (1.0f + e) : e / (1.0f + e);
      result = storage_round<T>(a * sigmoid) * b;
    } else {
      result = a + b;
    }
    store_elem(out, i, result);
  }
}

bool valid_dtype(int dtype) { return dtype == DL_BF16 || dtype == DL_F32; }

}  // namespace
}  // namespace dl

using dl::guard;
using dl::require;

extern "C" {

int dl_projection(dl_queue* queue, int dtype, const void* input, const void* weight, void* output,
                  uint64_t rows, uint64_t input_width, uint64_t output_width,
                  const uint64_t* output_position) {
  return guard([&] {
    dl::enter(queue);
    require(dl::valid_dtype(dtype), "unsupported storage type");
    require(input && weight && output, "null operand");
    require(rows > 0 && input_width > 0 && output_width > 0, "empty projection");
    if (dtype == DL_BF16)
      dl::launch_projection_rowmajor<uint16_t>(queue->stream, input, weight, output, rows, input_width,
                                               output_width, output_position);
    else
      dl::launch_projection_rowmajor<float>(queue->stream, input, weight, output, rows, input_width,
                                            output_width, output_position);
    dl::check_launch(queue, "projection");
  });
}

int dl_rms_norm(dl_queue* queue, int dtype, const void* input, const void* weight, void* output,
                uint64_t rows, uint64_t width, float epsilon) {
  return guard([&] {
    dl::enter(queue);
    require(dl::valid_dtype(dtype), "unsupported storage type");
    require(input && weight && output, "null operand");
    require(rows > 0 && width > 0, "empty normalization");
    require(epsilon > 0.0f, "epsilon must be positive");
    const unsigned grid = dl::grid_for(rows, 1, 65535);
    auto run = [&](auto tag, auto wide) {
      using T = decltype(tag);
      dl::rms_norm_rows<T, decltype(wide)::value><<<grid, dl::kThreads, 0, queue->stream>>>(
          static_cast<const T*>(input), static_cast<const T*>(weight), static_cast<T*>(output), rows, width, epsilon);
    };
    auto run_width = [&](auto tag) {
      if (width >= dl::kWideNorm)
        run(tag, std::true_type{});
      else
        run(tag, std::false_type{});
    };
    if (dtype == DL_BF16)
      run_width(uint16_t{});
    else
      run_width(float{});
    dl::check_launch(queue, "rms_norm");
  });
}

int dl_rotary(dl_queue* queue, int dtype, const void* input, void* output, uint64_t positions,
              uint64_t heads, uint64_t width, uint64_t first_position, double theta,
              const uint64_t* device_position, int positioned_output) {
  return guard([&] {
    dl::enter(queue);
    require(dl::valid_dtype(dtype), "unsupported storage type");
    require(input && output, "null operand");
    require(positions > 0 && heads > 0 && width > 0 && width % 2 == 0, "invalid rotary shape");
    require(theta > 0.0 && theta < 1e300, "theta must be positive and finite");
    const uint64_t pairs = positions * heads * (width / 2);
    const unsigned grid = dl::grid_for(pairs, dl::kThreads, 65535);
    if (dtype == DL_BF16)
      dl::rotary_pairs<uint16_t><<<grid, dl::kThreads, 0, queue->stream>>>(
          static_cast<const uint16_t*>(input), static_cast<uint16_t*>(output), pairs, heads, width,
          first_position, theta, device_position, positioned_output);
    else
      dl::rotary_pairs<float><<<grid, dl::kThreads, 0, queue->stream>>>(
          static_cast<const float*>(input), static_cast<float*>(output), pairs, heads, width,
          first_position, theta, device_position, positioned_output);
    dl::check_launch(queue, "rotary");
  });
}

int dl_attention_scale(dl_queue* queue, float* output, uint64_t width) {
  return guard([&] {
    dl::enter(queue);
    require(output != nullptr && width > 0, "invalid attention scale arguments");
    dl::attention_scale_kernel<<<1, 1, 0, queue->stream>>>(output, width);
    dl::check_launch(queue, "attention_scale");
  });
}

int dl_attention(dl_queue* queue, int dtype, const void* query, const void* key, const void* value,
                 void* output, uint64_t positions, uint64_t query_heads, uint64_t kv_heads,
                 uint64_t width, uint64_t first_position, const uint64_t* device_position,
                 uint64_t capacity, const float* scale) {
  return guard([&] {
    dl::enter(queue);
    require(dl::valid_dtype(dtype), "unsupported storage type");
    require(query && key && value && output && scale, "null operand");
    require(positions > 0 && query_heads > 0 && kv_heads > 0 && width > 0, "empty attention");
    require(query_heads % kv_heads == 0, "query heads must be a multiple of KV heads");
    const uint64_t keys = device_position ? capacity : first_position + positions;
    require(keys > 0, "no visible keys");
    const uint64_t shared_bytes = (width + keys) * sizeof(float);
    require(shared_bytes <= 160 * 1024 - 2 * 1024, "attention exceeds on-chip score storage",
            DL_LENGTH_ERROR);
    const uint64_t tasks = positions * query_heads;
    const unsigned grid = dl::grid_for(tasks, 1, 65535);
    const bool aligned = (reinterpret_cast<uintptr_t>(query) | reinterpret_cast<uintptr_t>(key) |
                          reinterpret_cast<uintptr_t>(value)) % 16 == 0;
    if (width == dl::kHeadWidth && aligned && query_heads <= UINT32_MAX) {
      auto run = [&](auto tag) {
        using T = decltype(tag);
        dl::attention_heads<T><<<grid, dl::kRowThreads, shared_bytes, queue->stream>>>(
            static_cast<const T*>(query), static_cast<const T*>(key), static_cast<const T*>(value),
            static_cast<T*>(output), tasks, static_cast<uint32_t>(query_heads), static_cast<uint32_t>(kv_heads),
            first_position, scale, device_position);
      };
      if (dtype == DL_BF16)
        run(uint16_t{});
      else
        run(float{});
    } else if (dtype == DL_BF16)
      dl::attention_retained<uint16_t><<<grid, dl::kThreads, shared_bytes, queue->stream>>>(
          static_cast<const uint16_t*>(query), static_cast<const uint16_t*>(key),
          static_cast<const uint16_t*>(value), static_cast<uint16_t*>(output), tasks, query_heads,
          kv_heads, width, first_position, scale, device_position);
    else
      dl::attention_retained<float><<<grid, dl::kThreads, shared_bytes, queue->stream>>>(
          static_cast<const float*>(query), static_cast<const float*>(key),
          static_cast<const float*>(value), static_cast<float*>(output), tasks, query_heads, kv_heads,
          width, first_position, scale, device_position);
    dl::check_launch(queue, "attention");
  });
}

int dl_embedding(dl_queue* queue, int dtype, const uint32_t* tokens, const void* weight,
                 void* output, uint64_t rows, uint64_t width, uint64_t vocabulary) {
  return guard([&] {
    dl::enter(queue);
    require(dl::valid_dtype(dtype), "unsupported storage type");
    require(tokens && weight && output, "null operand");
    require(rows > 0 && width > 0 && vocabulary > 0, "empty embedding");
    const unsigned grid = dl::grid_for(rows, 1, 65535);
    if (dtype == DL_BF16)
      dl::embedding_rows<uint16_t><<<grid, dl::kThreads, 0, queue->stream>>>(
          tokens, static_cast<const uint16_t*>(weight), static_cast<uint16_t*>(output), rows, width,
          vocabulary);
    else
      dl::embedding_rows<uint32_t><<<grid, dl::kThreads, 0, queue->stream>>>(
          tokens, static_cast<const uint32_t*>(weight), static_cast<uint32_t*>(output), rows, width,
          vocabulary);
    dl::check_launch(queue, "embedding");
  });
}

static int elementwise_entry(dl_queue* queue, int dtype, const void* left, const void* right,
                             void* output, uint64_t count, bool silu) {
  return guard([&] {
    dl::enter(queue);
    require(dl::valid_dtype(dtype), "unsupported storage type");
    require(left && right && output, "null operand");
    require(count > 0, "empty elementwise operation");
    const unsigned grid = dl::grid_for(count, dl::kThreads, 65535);
    hipStream_t s = queue->stream;
    if (dtype == DL_BF16) {
      auto l = static_cast<const uint16_t*>(left), r = static_cast<const uint16_t*>(right);
      auto o = static_cast<uint16_t*>(output);
      if (silu)
        dl::elementwise<uint16_t, true><<<grid, dl::kThreads, 0, s>>>(l, r, o, count);
      else
        dl::elementwise<uint16_t, false><<<grid, dl::kThreads, 0, s>>>(l, r, o, count);
    } else {
      auto l = static_cast<const float*>(left), r = static_cast<const float*>(right);
      auto o = static_cast<float*>(output);
      if (silu)
        dl::elementwise<float, true><<<grid, dl::kThreads, 0, s>>>(l, r, o, count);
      else
        dl::elementwise<float, false><<<grid, dl::kThreads, 0, s>>>(l, r, o, count);
    }
    dl::check_launch(queue, silu ? "silu_multiply" : "add");
  });
}

int dl_add(dl_queue* queue, int dtype, const void* left, const void* right, void* output,
           uint64_t count) {
  return elementwise_entry(queue, dtype, left, right, output, count, false);
}

int dl_silu_multiply(dl_queue* queue, int dtype, const void* gate, const void* up, void* output,
                     uint64_t count) {
  return elementwise_entry(queue, dtype, gate, up, output, count, true);
}

int dl_gather_rows(dl_queue* queue, const void* input, void* output, uint64_t row_bytes,
                   const uint64_t* rows, uint64_t count) {
  return guard([&] {
    dl::enter(queue);
    require(input && output && (rows || count == 0), "null operand");
    require(row_bytes > 0, "empty rows");
    for (uint64_t i = 0; i < count; ++i) {
      dl::check_hip(hipMemcpyAsync(static_cast<char*>(output) + i * row_bytes,
                                   static_cast<const char*>(input) + rows[i] * row_bytes, row_bytes,
                                   hipMemcpyDeviceToDevice, queue->stream),
                    "gather rows");
    }
  });
}

}  // extern "C"
