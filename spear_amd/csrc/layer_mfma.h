// A product of a few rows with weights as they lie, for the layer's kernels at sizes where launches and latency count: 16 kW
// weight rows by 16 kNT rows of x, a quarter of the columns per wavefront, on v_mfma_f32_16x16x32_bf16. The weights
// are the A operand, the rows of x the B operand; both come from memory as the matrix unit wants them, 8 consecutive columns per
// lane, without LDS. In the result tile, lane 16 q + n has the weight rows 4 q .. 4 q + 3 of row n of x.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace spear_btp {

namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x4_t mfma(uint4 a, uint4 b, f32x4_t acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), acc, 0, 0, 0);
}

constexpr int kStep = 32;  // columns of one matrix instruction
constexpr int kParts = 4;  // wavefronts of a workgroup: quarters of the columns

// Matrix instructions along a quarter of K columns (the last quarter may have fewer).
__host__ __device__ inline int quarter_steps(int K) { return ((K + kStep - 1) / kStep + kParts - 1) / kParts; }

template <int kNT, int kChunk, int kW>
struct Operands {
  uint4 w[kChunk][kW];
  uint4 x[kChunk][kNT];
};

// acc[i][t] <- w[i] x[t] over the columns of `wave`'s quarter. w[i], x[t]: this lane's row (lane % 16) of the tile, K columns, 16-byte
// aligned, K a multiple of 8 and at least 8. The loads of kChunk steps of 32 columns are in flight while the chunk before is multiplied.
template <int kNT, int kChunk, int kW>
__device__ __forceinline__ void quarter_product(const uint16_t* const (&w)[kW], const uint16_t* const (&x)[kNT], int K, int wave, int q,
                                                f32x4_t (&acc)[kW][kNT]) {
#pragma unroll
  for (int t = 0; t < kNT; ++t) {
#pragma unroll
    for (int i = 0; i < kW; ++i) acc[i][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  }
  const int steps = (K + kStep - 1) / kStep, share = quarter_steps(K);
  const int from = wave * share, to = min(from + share, steps);
  auto load = [&](Operands<kNT, kChunk, kW>& o, int s0) {
#pragma unroll
    for (int s = 0; s < kChunk; ++s) {
      const int k = min((s0 + s) * kStep + 8 * q, K - 8);  // K is a multiple of 8; what lies past it is replaced by zeros below
#pragma unroll
      for (int i = 0; i < kW; ++i) o.w[s][i] = *reinterpret_cast<const uint4*>(w[i] + k);
#pragma unroll
      for (int t = 0; t < kNT; ++t) o.x[s][t] = *reinterpret_cast<const uint4*>(x[t] + k);
    }
  };
  auto multiply = [&](Operands<kNT, kChunk, kW>& o, int s0) {
#pragma unroll
    for (int s = 0; s < kChunk; ++s) {
      const int k = (s0 + s) * kStep;
      if (s0 + s >= to) break;
      if (k + kStep > K && k + 8 * q >= K) {
        const uint4 zero = make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < kW; ++i) o.w[s][i] = zero;
#pragma unroll
        for (int t = 0; t < kNT; ++t) o.x[s][t] = zero;
      }
#pragma unroll
      for (int t = 0; t < kNT; ++t) {
#pragma unroll
        for (int i = 0; i < kW; ++i) acc[i][t] = mfma(o.w[s][i], o.x[s][t], acc[i][t]);
      }
    }
  };
  Operands<kNT, kChunk, kW> even, odd;
  if (from < to) load(even, from);

  for (int s = from; s < to; s += 2 * kChunk) {
    if (s + kChunk < to) load(odd, s + kChunk);
    multiply(even, s);
    if (s + 2 * kChunk < to) load(even, s + 2 * kChunk);
    if (s + kChunk < to) multiply(odd, s + kChunk);
  }
}

// The four wavefronts' parts of the tiles added up through LDS: sum[i] of token tile `wave` in wavefront `wave` (< kNT). Every
// thread of the workgroup has to call it.
template <int kNT, int kW>
__device__ __forceinline__ void add_quarters(f32x4_t (&partial)[kParts][kW][kNT][64], const f32x4_t (&acc)[kW][kNT], int wave, int lane,
                                             f32x4_t (&sum)[kW]) {
#pragma unroll
  for (int t = 0; t < kNT; ++t) {
#pragma unroll
    for (int i = 0; i < kW; ++i) partial[wave][i][t][lane] = acc[i][t];
  }
  __syncthreads();
  if (wave >= kNT) return;
#pragma unroll
  for (int i = 0; i < kW; ++i) {
    sum[i] = partial[0][i][wave][lane];
#pragma unroll
    for (int w = 1; w < kParts; ++w) sum[i] += partial[w][i][wave][lane];
  }
}

}  // namespace

}  // namespace spear_btp
