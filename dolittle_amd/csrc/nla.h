// Vector operations of the NLA injection and steering protocol on gfx950:
// the injection normalization (src/kernels/cuda/injection.cu:49-98, law H2
// of docs/architecture/execution-boundary.md:489-498), the steering direction
// (src/kernels/cuda/steering.cu:69-100) and the one-row residual intervention
// (steering.cu:107-159).  Each runs as one workgroup: eight lanes of the first
// wavefront hold the eight strided FP32 square sums, thread 0 combines them,
// and the whole workgroup applies the row update.
#pragma once

#include "dl_device.h"

namespace dl::nla {

constexpr unsigned kLanes = 8;      // strided partial sums of the reference reduction
constexpr unsigned kThreads = 256;  // one workgroup per vector operation

constexpr uint64_t kChunk = 4096;   // squares in LDS at a time
constexpr int kBatch = 8;           // values a thread has in flight

// f(i, load(i)) for the indices i = first + threadIdx.x + k * blockDim.x below
// `end`, kBatch loads ahead of the calls that use them.
template <class Load, class F>
__device__ __forceinline__ void for_each_loaded(uint64_t first, uint64_t end, Load&& load, F&& f) {
  for (uint64_t base = first + threadIdx.x; base < end; base += kBatch * blockDim.x) {
    decltype(load(base)) v[kBatch];
#pragma unroll
    for (int k = 0; k < kBatch; ++k) {
      const uint64_t i = base + k * blockDim.x;
      v[k] = load(i < end ? i : base);
    }
#pragma unroll
    for (int k = 0; k < kBatch; ++k) {
      const uint64_t i = base + k * blockDim.x;
      if (i < end) f(i, v[k]);
    }
  }
}

// sum_i value(i)^2 in the reference order: lane k < 8 accumulates
// i = k, k + 8, k + 16, ... ascending, with separately rounded multiply and
// add; thread 0 then adds lanes 0..7 left to right.  Every thread of the
// workgroup calls; all receive the sum (kept in sums[kLanes]).  The whole
// workgroup loads and squares into LDS and the eight lanes only add from
// there, 16 reads ahead (with eight threads loading as they add, a 4096-wide
// row waited for 512 memory latencies in turn: 40-56 us per operation, now
// 8).  value(load(i)) may have side effects: it runs once per index.
template <class Load, class F>
__device__ __forceinline__ float square_sum(uint64_t width, Load&& load, F&& value, float* sums) {
  __shared__ float squares[kChunk];
  float sum = 0.0f;
  for (uint64_t base = 0; base < width; base += kChunk) {
    const int n = static_cast<int>(width - base < kChunk ? width - base : kChunk);
    for_each_loaded(base, base + n, load, [&](uint64_t i, auto raw) {
      const float v = value(raw);
      squares[i - base] = __fmul_rn(v, v);
    });
    __syncthreads();
    if (threadIdx.x < kLanes) {
      constexpr int kAhead = 16;
      int i = threadIdx.x;
      for (; i + (kAhead - 1) * static_cast<int>(kLanes) < n; i += kAhead * kLanes) {
        float s[kAhead];
#pragma unroll
        for (int k = 0; k < kAhead; ++k) s[k] = squares[i + k * kLanes];
#pragma unroll
        for (int k = 0; k < kAhead; ++k) sum = __fadd_rn(sum, s[k]);
      }
      for (; i < n; i += kLanes) sum = __fadd_rn(sum, squares[i]);
    }
    __syncthreads();
  }
  if (threadIdx.x < kLanes) sums[threadIdx.x] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    float total = 0.0f;
    for (unsigned k = 0; k < kLanes; ++k) total = __fadd_rn(total, sums[k]);
    sums[kLanes] = total;
  }
  __syncthreads();
  return sums[kLanes];
}

__device__ __forceinline__ bool finite(float v) { return __builtin_isfinite(v); }

// The intervention's row update (steering.cu:107-159) on one row of width
// `width`: state[0] is the status latch, state[1] the application count.  A
// row already intervened on (count nonzero) or a prior failure makes this
// application invalid (the row is left unchanged, the count still grows).
// beta = strength * sqrt(sum h^2); h[i] = narrow(h[i] + beta * u[i]) with
// separate rounding; a nonfinite beta or stored value latches status.
// `sums` holds kLanes + 2 floats and `invalid` one word of LDS.
template <class T>
__device__ __forceinline__ void intervene_row(T* row, const float* direction, uint32_t* state, uint64_t width,
                                              float strength, float* sums, uint32_t* invalid) {
  if (threadIdx.x == 0) {
    *invalid = (state[0] != 0 || state[1] != 0) ? 1u : 0u;
    state[1] = state[1] + 1;
  }
  __syncthreads();
  auto load = [&](uint64_t i) { return load_elem(row, i); };
  const float sum = square_sum(width, load, [](float v) { return v; }, sums);
  if (threadIdx.x == 0) {
    const float beta = __fmul_rn(strength, __builtin_sqrtf(sum));
    sums[kLanes + 1] = beta;
    if (!finite(beta)) *invalid = 1u;
  }
  __syncthreads();
  const float beta = sums[kLanes + 1];
  const bool valid = *invalid == 0;
  __syncthreads();
  if (valid) {
    for_each_loaded(
        0, width, [&](uint64_t i) { return float2{load_elem(row, i), direction[i]}; },
        [&](uint64_t i, float2 v) {
          const float value = __fadd_rn(v.x, __fmul_rn(beta, v.y));
          store_elem(row, i, value);
          if (!finite(value) || !finite(storage_round<T>(value))) atomicOr(invalid, 1u);
        });
  }
  __syncthreads();
  if (threadIdx.x == 0) state[0] = *invalid;
}

}  // namespace dl::nla
