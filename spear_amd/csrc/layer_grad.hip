// The small passes around the matrix products of a Phalanx layer's backward on gfx950 (MI355X).
//
// layer_sums: column sums of several fp32 arrays, rounded to 16 bits, in one launch. They are the weight gradients' partial
// products (one per slice of the token axis: few rows, millions of columns) and the bias gradients' partial sums (one per
// 64 time steps of a batch row: thousands of rows, a few hundred columns). Both are bound by reading the fp32 array once. As
// library reductions and conversions they were ten launches: at B=1024 L=128 dim=512 101 us of GPU time for 123 MB, most of it in
// the tall arrays and in passes over results that had just been written; here 37 us.
//
// layer_stack: the projections' weights one under the other in the column order of the packed gradient buffer, zero rows for its
// padding columns, and zeros in those columns: one launch where a concatenation and two fills were three (and a copy more where a
// weight's type or layout had to be changed). Bound by the launch at small sizes, by writing [ld, K] else.
//
// layer_transpose: the same weights and proj_out's as the large-tile kernel (layer_gemm.hip) wants them for the input gradients, rows of the
// reduction's columns, and the same zeros. 64 x 64 tiles through LDS, 16 bytes per access on both sides; bound by the launch at small
// sizes (6 us for 2.6 MB at dim 512), by reading and writing each weight once else.
//
// The parts of layer_wgrad come as its accumulators lie and are put in order on the way out (8-byte stores, 32 bytes in a row).
//
// A block of layer_sums, 512 threads, takes either 2048 columns, four to a thread, and walks the rows with eight 16-byte loads in flight
// (few rows), or 16 columns with 32 threads to a column that add up through LDS (many rows: 2048 rows by 512 columns
// still make 32 blocks). Sums are taken in an order that depends on the shape only: the same bits in every run.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "btp_device.h"
#include "btp_launch.h"

namespace spear_btp {

namespace {

constexpr int kThreads = 512;
constexpr int kFlatColumns = 4 * kThreads;
constexpr int kTallColumns = 16, kTallLanes = kThreads / kTallColumns;

// Four columns to a thread need rows that start on 16 bytes and enough columns to fill the chip; with 64 rows or fewer the
// weight gradients' arrays all have them. Narrow ones go the tall way at any number of rows.
__host__ __device__ inline bool is_flat(const LayerSumJob& j) { return j.cols % 4 == 0 && j.rows <= 64; }

// A job over the parts of layer_wgrad: four consecutive columns of one row of the result to a thread.
constexpr int kTileQuads = kWgradSide * kWgradSide / 4;

inline long job_blocks(const LayerSumJob& j) {
  if (j.splits > 0) return (long)((j.rows + kWgradSide - 1) / kWgradSide) * ((j.cols + kWgradSide - 1) / kWgradSide) * (kTileQuads / kThreads);
  return is_flat(j) ? (j.cols + kFlatColumns - 1) / kFlatColumns : (j.cols + kTallColumns - 1) / kTallColumns;
}

struct Jobs {
  LayerSumJob job[kLayerSumJobs];
  long first_block[kLayerSumJobs + 1];
};

template <class E>
__global__ __launch_bounds__(kThreads) void layer_sums_kernel(const Jobs jobs, int n) {
  __shared__ float part[kTallLanes][kTallColumns];
  int at = 0;
  while (at + 1 < n && (long)blockIdx.x >= jobs.first_block[at + 1]) ++at;
  const LayerSumJob j = jobs.job[at];
  const long block = (long)blockIdx.x - jobs.first_block[at];
  if (j.splits > 0) {
    constexpr int kBlocks = kTileQuads / kThreads;
    const int tile = (int)(block / kBlocks), e = (int)(block % kBlocks) * kThreads + (int)threadIdx.x;
    const int tiles_n = (int)((j.rows + kWgradSide - 1) / kWgradSide), tiles = tiles_n * (int)((j.cols + kWgradSide - 1) / kWgradSide);
    const int k0 = tile / tiles_n * kWgradSide, n0 = tile % tiles_n * kWgradSide;
    // where layer_wgrad's accumulators lie: wavefront, tile of dy's columns, tile of x's columns, lane
    const int wave = e >> 11, i = (e >> 8) & 7, jt = (e >> 6) & 3, lane = e & 63, wn = wave & 3;
    const bool full = j.cols - k0 > 128;
    const int n = n0 + 128 * (wave >> 2) + 16 * i + (lane & 15), k = k0 + 16 * ((full ? 4 : 2) * wn + jt) + 4 * (lane >> 4);
    if ((!full && jt >= 2) || n >= j.rows || k >= j.cols) return;
    const float* p = j.in + ((long)tile * kTileQuads + e) * 4;
    const long split = (long)tiles * kTileQuads * 4;
    float4 sum = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    int row = 0;
    for (; row + 8 <= j.splits; row += 8) {
      float4 q[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) q[u] = *reinterpret_cast<const float4*>(p + (row + u) * split);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        sum.x += q[u].x; sum.y += q[u].y; sum.z += q[u].z; sum.w += q[u].w;
      }
    }
    for (; row < j.splits; ++row) {
      const float4 q = *reinterpret_cast<const float4*>(p + row * split);
      sum.x += q.x; sum.y += q.y; sum.z += q.z; sum.w += q.w;
    }
    *reinterpret_cast<uint2*>(j.out + (long)n * j.cols + k) = make_uint2(E::pack2(sum.x, sum.y), E::pack2(sum.z, sum.w));
    return;
  }
  if (is_flat(j)) {
    const long col = block * kFlatColumns + 4 * (long)threadIdx.x;
    if (col >= j.cols) return;
    const float* p = j.in + col;
    float4 sum = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    int row = 0;
    for (; row + 8 <= j.rows; row += 8) {
      float4 q[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) q[i] = *reinterpret_cast<const float4*>(p + (long)(row + i) * j.cols);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        sum.x += q[i].x; sum.y += q[i].y; sum.z += q[i].z; sum.w += q[i].w;
      }
    }
    for (; row < j.rows; ++row) {
      const float4 q = *reinterpret_cast<const float4*>(p + (long)row * j.cols);
      sum.x += q.x; sum.y += q.y; sum.z += q.z; sum.w += q.w;
    }
    *reinterpret_cast<uint2*>(j.out + col) = make_uint2(E::pack2(sum.x, sum.y), E::pack2(sum.z, sum.w));
    return;
  }
  const int lane = threadIdx.x / kTallColumns, c = threadIdx.x % kTallColumns;
  const long col = block * kTallColumns + c;
  float sum = 0.0f;
  if (col < j.cols) {
    const float* p = j.in + col;
    long row = lane;
    for (; row + 7 * kTallLanes < j.rows; row += 8 * kTallLanes) {
      float q[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) q[i] = p[(row + i * kTallLanes) * j.cols];
#pragma unroll
      for (int i = 0; i < 8; ++i) sum += q[i];
    }
    for (; row < j.rows; row += kTallLanes) sum += p[row * j.cols];
  }
  part[lane][c] = sum;
  __syncthreads();
  if (lane == 0 && col < j.cols) {
    for (int i = 1; i < kTallLanes; ++i) sum += part[i][c];
    j.out[col] = (uint16_t)E::pack2(sum, 0.0f);
  }
}

// The 16-byte pieces of packed's rows that reach past its last used column <- zeros from that column on. i: which of them.
__device__ __forceinline__ void clear_padding(uint16_t* packed, int used, int ld, long i) {
  const int first = used / 8, per_row = ld / 8 - first;
  const long row = i / per_row;
  const int col = 8 * (first + (int)(i - row * per_row));
  uint16_t* at = packed + row * ld + col;
  if (col >= used) {
    *reinterpret_cast<uint4*>(at) = make_uint4(0, 0, 0, 0);
  } else {
    for (int e = used - col; e < 8; ++e) at[e] = 0;
  }
}

// One 16-byte piece per thread: first the pieces of the stacked weights [ld, K], then those of the buffer's rows that reach
// past the last used column. Only columns from `used` on are written there.
__global__ __launch_bounds__(256) void layer_stack_kernel(const LayerStackArgs p, long stack_pieces, long total) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const uint4 zero = make_uint4(0, 0, 0, 0);
  if (i < stack_pieces) {
    const int per_row = p.K / 8;
    long row = i / per_row;
    const int piece = (int)(i - row * per_row);
    uint4 q = zero;
    for (int part = 0; part < 4; ++part) {
      if (row < p.rows[part]) {
        q = *reinterpret_cast<const uint4*>(p.weight[part] + row * p.K + 8 * piece);
        break;
      }
      row -= p.rows[part];
    }
    *reinterpret_cast<uint4*>(p.stacked + i * 8) = q;
    return;
  }
  clear_padding(p.packed, p.used, p.ld, i - stack_pieces);
}

struct Transposes {
  LayerTransposeJob job[kLayerTransposeJobs];
  int first_block[kLayerTransposeJobs + 1];
};

constexpr int kSide = 64;

__global__ __launch_bounds__(256) void layer_transpose_kernel(const Transposes jobs, int n, uint16_t* packed, int used, int ld, long pieces) {
  __shared__ __attribute__((aligned(16))) uint16_t tile[kSide][kSide + 8];
  if ((int)blockIdx.x >= jobs.first_block[n]) {
    const long i = (long)((int)blockIdx.x - jobs.first_block[n]) * 256 + threadIdx.x;
    if (i < pieces) clear_padding(packed, used, ld, i);
    return;
  }
  int at = 0;
  while ((int)blockIdx.x >= jobs.first_block[at + 1]) ++at;
  const LayerTransposeJob j = jobs.job[at];
  const int block = (int)blockIdx.x - jobs.first_block[at], across = (j.cols + kSide - 1) / kSide;
  const int r0 = block / across * kSide, c0 = block % across * kSide;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = (int)threadIdx.x / 8 + 32 * i, c = (int)threadIdx.x % 8 * 8;
    uint4 q = make_uint4(0, 0, 0, 0);
    if (r0 + r < j.rows && c0 + c < j.cols) q = *reinterpret_cast<const uint4*>(j.in + (long)(r0 + r) * j.cols + c0 + c);
    *reinterpret_cast<uint4*>(&tile[r][c]) = q;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c = (int)threadIdx.x / 8 + 32 * i, r = (int)threadIdx.x % 8 * 8;
    if (c0 + c >= j.cols || r0 + r >= j.width) continue;
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = tile[r + 2 * e][c] | (uint32_t)tile[r + 2 * e + 1][c] << 16;
    *reinterpret_cast<uint4*>(j.out + (long)(c0 + c) * j.ld + r0 + r) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

}  // namespace

hipError_t layer_transpose(const LayerTransposeJob* jobs, int n, uint16_t* packed, long M, int used, int ld, hipStream_t s) {
  Transposes all{};
  long blocks = 0;
  for (int i = 0; i < n; ++i) {
    all.job[i] = jobs[i];
    all.first_block[i] = (int)blocks;
    blocks += (long)((jobs[i].width + kSide - 1) / kSide) * ((jobs[i].cols + kSide - 1) / kSide);
  }
  all.first_block[n] = (int)blocks;
  const long pieces = used < ld ? M * (ld / 8 - used / 8) : 0;
  blocks += (pieces + 255) / 256;
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(layer_transpose_kernel, dim3((unsigned)blocks), dim3(256), 0, s, all, n, packed, used, ld, pieces);
  return hipGetLastError();
}

hipError_t layer_stack(const LayerStackArgs& p, hipStream_t s) {
  const long stack_pieces = (long)p.ld * (p.K / 8), total = stack_pieces + (p.used < p.ld ? p.M * (p.ld / 8 - p.used / 8) : 0);
  if (total == 0) return hipSuccess;
  hipLaunchKernelGGL(layer_stack_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, p, stack_pieces, total);
  return hipGetLastError();
}

long layer_sums_blocks(const LayerSumJob* jobs, int n) {
  long blocks = 0;
  for (int i = 0; i < n; ++i) blocks += job_blocks(jobs[i]);
  return blocks;
}

hipError_t layer_sums(const LayerSumJob* jobs, int n, int dtype, hipStream_t s) {
  Jobs all{};
  long blocks = 0;
  for (int i = 0; i < n; ++i) {
    all.job[i] = jobs[i];
    all.first_block[i] = blocks;
    blocks += job_blocks(jobs[i]);
  }
  all.first_block[n] = blocks;
  if (blocks == 0) return hipSuccess;
  if (dtype == kBf16) hipLaunchKernelGGL(layer_sums_kernel<Bf16>, dim3((unsigned)blocks), dim3(kThreads), 0, s, all, n);
  else hipLaunchKernelGGL(layer_sums_kernel<Fp16>, dim3((unsigned)blocks), dim3(kThreads), 0, s, all, n);
  return hipGetLastError();
}

}  // namespace spear_btp
