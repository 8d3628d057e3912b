// The layer's linear projections at sizes where launches count, on gfx950 (MI355X): up to four of them on the same rows in one
// launch.
//
//     out_j[M, N_j] = x[M, K] w_j[N_j, K]^T + bias_j          bf16, fp32 sums, rounded once
//
// The four input projections of a thousand tokens are a GFLOP or two. The library serves them one by one, in 5 to 7 us each on
// the GPU and about 15 us of host time per call, which is what such a layer is bound by. A workgroup makes 16 kW columns by 16 kNT
// rows (layer_mfma.h: a quarter of K per wavefront), whatever array the columns belong to, so the narrow arrays share the chip with the
// wide ones.
//
// Longer inputs are for the tiles of layer_gemm.hip (`fastest`). One projection (dim x dim) here / as the library's
// product, us in a HIP graph: M=1 dim=512 2.9 / 3.7, dim=2048 4.7 / 5.2; M=16 dim=512 3.3 / 3.8, dim=1024 4.3 / 4.3, dim=2048 6.0 / 5.3; M=64 dim=1024 4.4 /
// 6.5, dim=2048 7.9 / 7.4; M=128 dim=768 5.2 / 4.7, dim=1024 5.4 / 5.2, dim=2048 9.6 / 6.7. As a call the library's product costs the host 15 us more.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "btp_device.h"
#include "btp_launch.h"
#include "layer_mfma.h"

namespace spear_btp {

namespace {

template <int kNT, int kChunk, int kW>
__global__ __launch_bounds__(256) void layer_linear_kernel(const LayerLinearArgs p, int groups) {
  constexpr int kCols = 16 * kW;
  __shared__ f32x4_t partial[kParts][kW][kNT][64];
  const int lane = threadIdx.x & 63, n = lane & 15, q = lane >> 4, wave = threadIdx.x >> 6;
  int group = (int)(blockIdx.x % (unsigned)groups), j = 0;
  const int first = (int)(blockIdx.x / (unsigned)groups) * 16 * kNT;
  while (group >= (p.N[j] + kCols - 1) / kCols) group -= (p.N[j++] + kCols - 1) / kCols;
  const int N = p.N[j], col = kCols * group, K = p.K;
  const uint16_t *w[kW], *x[kNT];
#pragma unroll
  for (int i = 0; i < kW; ++i) w[i] = p.w[j] + (long)min(col + 16 * i + n, N - 1) * K;  // past the last row or column: read it, store nothing
#pragma unroll
  for (int t = 0; t < kNT; ++t) x[t] = p.x + (long)min(first + 16 * t + n, p.M - 1) * p.ldx;
  f32x4_t acc[kW][kNT], sum[kW];
  quarter_product<kNT, kChunk, kW>(w, x, K, wave, q, acc);
  add_quarters<kNT, kW>(partial, acc, wave, lane, sum);
  const int row = first + 16 * wave + n;
  if (wave >= kNT || row >= p.M) return;
  if (p.pos != nullptr && blockIdx.x % (unsigned)groups == 0 && q == 0) {  // one lane of the grid per row
    const int next = p.pos[row] + 1;
    p.pos[row] = next >= p.block_len ? 0 : next;
  }
  const uint16_t* bias = p.bias[j];
  uint16_t* out = p.out[j] + (long)row * N;
#pragma unroll
  for (int i = 0; i < kW; ++i) {
    const int c = col + 16 * i + 4 * q;
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = sum[i][e] + (bias != nullptr && c + e < N ? Bf16::lo(bias[c + e]) : 0.0f);
    const uint2 packed = make_uint2(Bf16::pack2(v[0], v[1]), Bf16::pack2(v[2], v[3]));
    if (N % 4 == 0) {  // rows of the result start on 8 bytes and end with a whole piece
      if (c < N) *reinterpret_cast<uint2*>(out + c) = packed;
    } else {
      if (c < N) out[c] = (uint16_t)packed.x;
      if (c + 1 < N) out[c + 1] = (uint16_t)(packed.x >> 16);
      if (c + 2 < N) out[c + 2] = (uint16_t)packed.y;
      if (c + 3 < N) out[c + 3] = (uint16_t)(packed.y >> 16);
    }
  }
}

template <int kNT, int kChunk, int kW>
void launch(const LayerLinearArgs& p, long groups, hipStream_t s) {
  const long tiles = (p.M + 16 * kNT - 1) / (16 * kNT);
  hipLaunchKernelGGL((layer_linear_kernel<kNT, kChunk, kW>), dim3((unsigned)(groups * tiles)), dim3(256), 0, s, p, (int)groups);
}

// Tiles of `cols` columns that the arrays of a call have.
long groups_of(const LayerLinearArgs& p, int cols) {
  long groups = 0;
  for (int j = 0; j < p.jobs; ++j) groups += (p.N[j] + cols - 1) / cols;
  return groups;
}

// The instance of the kernel here for a call, 16 kNT rows by 16 kW columns to a workgroup, and its time in us as fitted to their times at K = 256 to
// 4096. The smallest tile of which each compute unit gets one at most: its operands are the longest part of its time. [M, K] x [K, K], the instance that
// the rule takes / the next larger tile, us: M=16 K=512 3.3 / 3.8, K=1024 4.3 / 5.3, K=2048 6.0 / 7.8, K=4096 10.1 / 13.6 (64 columns 4.9, 7.3, 11.6, 21.0); M=64
// K=2048 7.9 / 9.6 (16 columns 9.5); M=128 K=2048 9.6 / 11.7.
struct Instance {
  int rows, cols;
  double us;
};

Instance instance(const LayerLinearArgs& p) {
  const double K = p.K;
  const long g16 = groups_of(p, 16), g32 = groups_of(p, 32), g64 = groups_of(p, 64), r16 = (p.M + 15l) / 16, r32 = (p.M + 31l) / 32, r64 = (p.M + 63l) / 64;
  if (g16 * r16 <= 256) return {16, 16, 2.2 + 0.0019 * K};
  if (g32 * r16 <= 256) return {16, 32, 2.7 + 0.0026 * K};
  if (g32 * r32 <= 256) return {32, 32, 2.8 + 0.0035 * K};
  if (g64 * r16 <= 256) return {16, 64, 3.6 + 0.0041 * K};
  if (g64 * r16 <= 512) return {32, 64, 3.5 + 0.0051 * K};
  return {64, 64, 3.7 + (double)((g64 * r64 + 255) / 256) * (0.5 + 0.0072 * K)};
}

}  // namespace

// Which kernel is the fastest, by their times in us as fitted to 56 shapes (dim 128 to 2048, 256 to 16384 rows) for the tiles: of 128 x 128, 0.47 us per
// 64 columns of K while each compute unit has one, twice that for two; of 256 x 256, 1 us. Four projections, dim = K, here / 128 / 256: K=128
// 1024 rows 5.0 / 5.2 / 9.1, 8192 rows 12.5 / 6.1 / 9.9; K=512 256 rows 5.7 / 7.9 / 16.2, 1024 rows 11.9 / 8.6 / 16.8, 8192 rows 56 / 21 / 19; K=1024 256 rows
// 10.7 / 11.6 / 24, 2048 rows 61 / 20 / 28, 4096 rows 106 / 36 / 29; K=2048 128 rows 17.7 / 18.6, 1024 rows 111 / 34 / 46; K=4096 1 row 18.6 / 36, 128 rows 60 / 33.
enum class Kernel { kHere, kMid, kLarge };

static Kernel fastest(const LayerLinearArgs& p) {
  if (!layer_gemm_takes(p)) return Kernel::kHere;
  auto tiles = [&](long side) { return groups_of(p, (int)side) * ((p.M + side - 1) / side); };
  const int steps = (p.K + 63) / 64;
  const long small_tiles = tiles(128);
  const double here = instance(p).us;
  const double mid = 4.2 + steps * (small_tiles <= 256 ? 0.47 : 1.0 * (double)((small_tiles + 511) / 512));
  const double large = 8.0 + (double)((tiles(256) + 255) / 256) * (1.0 + steps);
  if (p.pos != nullptr) return here <= mid ? Kernel::kHere : Kernel::kMid;  // the large tiles move no positions
  return here <= mid && here <= large ? Kernel::kHere : mid <= large ? Kernel::kMid : Kernel::kLarge;
}

// Up to here 128 x 128 tiles add up K in the four quarters that the kernel here has in four wavefronts: a call of such a size gives the same
// bits whichever of the two it goes to, and loses nothing against the shorter chains (of [2048, 1024] x [1024, 1024] 9.2e-5 of the
// results are not the nearest 16-bit value in quarters, 1.1e-4 in one chain over K). It takes 0.4 to 1.4 us more (a layer's forward at 1024
// rows, dim 512, 21.4 / 20.7 us; 4096 rows, 256, 21.5 / 20.1). Larger calls are added up in one chain by tiles of either size, as the library does.
static bool few(const LayerLinearArgs& p) {
  long columns = 0;
  for (int j = 0; j < p.jobs; ++j) columns += p.N[j];
  return p.jobs > 1 ? p.M * columns * p.K <= 1600000000 : p.K <= 512 && p.M * columns * p.K <= 300000000;
}

int layer_linear_choice(const LayerLinearArgs& p) { return (int)fastest(p); }

hipError_t layer_linear(const LayerLinearArgs& p, hipStream_t s) {
  if (p.jobs == 0 || p.M == 0) return hipSuccess;
  if (const Kernel k = fastest(p); k != Kernel::kHere) return layer_gemm(p, k == Kernel::kMid ? LayerTiles::kMid : LayerTiles::kLarge, few(p), s);
  const Instance at = instance(p);
  const long groups = groups_of(p, at.cols);
  if (at.cols == 16) launch<1, 4, 1>(p, groups, s);
  else if (at.cols == 32 && at.rows == 16) launch<1, 4, 2>(p, groups, s);
  else if (at.cols == 32) launch<2, 4, 2>(p, groups, s);
  else if (at.rows == 16) launch<1, 4, 4>(p, groups, s);
  else if (at.rows == 32) launch<2, 4, 4>(p, groups, s);
  else launch<4, 2, 4>(p, groups, s);
  return hipGetLastError();
}

}  // namespace spear_btp
