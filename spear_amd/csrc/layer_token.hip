// One decode token through the front of a Phalanx layer on gfx950 (MI355X): the four input projections and the mixing
// stage's step, in one launch.
//
//     a = x W_a^T + b_a   b = x W_b^T + b_b   c = x W_c^T + b_c   v = x W_v^T
//     A = sigmoid(a), h = A h + sigmoid(b) v, r = A r, out = (h + r c_prev) c + v      (phalanx_mix_step_kernel)
//
// In the reference this is four linear layers and step_jagged (spear/nn/phalanx/swr.py:166-221,
// spear/nn/phalanx/inference.py:178-278). One token per sequence is a few GFLOP at most: as four library products and a step it
// is bound by launches on the host and by the latency of short kernels on the GPU.
//
// A workgroup owns ONE head and 16 kNT tokens; its four wavefronts take a quarter of the columns each and add up through LDS, so
// the serial chain of loads is K / 4 columns long (with the columns of a head in one wavefront 28 us at B=1, 128 heads, against
// 11). The weights are the A operand of v_mfma_f32_16x16x32_bf16 (rows: the 16 features of the head's v, b and c, and the
// head's row of W_a sixteen times over), the tokens are the B operand: the result tiles of v, b, c and a then hold the same
// (feature, token) pair in the same lane and register and the step needs no exchange. Lane 16 q + n has the features
// 4 q .. 4 q + 3 of token n. Both operands come from memory as the matrix unit wants them (8 consecutive k per lane). The
// sums, the biases and the step stay in fp32 (the library products round a, b, c and v to 16 bits in between). The loads of
// `kChunk` steps of 32 columns are in flight while the chunk before is multiplied. Neighbouring workgroups take other heads, so an
// XCD's L2 sees an eighth of the weights where 8 divides the heads.
//
// Measured in a HIP graph, us, this kernel / four library products and the step kernel: B=1 8 heads 5.5 / 23.8, B=1 128 heads
// 10.8 / 30.1, B=256 32 heads 7.7 / 25.7, B=1024 32 heads 14.0 / 25.8 (1.7 GFLOP), B=1024 64 heads 33.7 / 43.0, 128 heads 111 / 64:
// every workgroup reads its weights and tokens through L2 once, which the library's larger tiles do less often, so the caller
// takes the library from B H K > 2^26 on. The whole step as a call at B=1024, 32 heads: 122 -> 23 us, with
// the output projection in layer_linear.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "btp_device.h"
#include "btp_launch.h"
#include "layer_mfma.h"

namespace spear_btp {

namespace {

__device__ __forceinline__ float sigmoid(float z) { return __builtin_amdgcn_rcpf(1.0f + __expf(-z)); }

template <int kNT, int kChunk>
__global__ __launch_bounds__(256) void layer_token_kernel(const LayerTokenArgs p) {
  // [wavefront][v, b, c, a][token tile][lane]: the partial sums of each wavefront's columns
  __shared__ f32x4_t partial[kParts][4][kNT][64];
  const int lane = threadIdx.x & 63, n = lane & 15, q = lane >> 4, wave = threadIdx.x >> 6;
  const int head = (int)(blockIdx.x % (unsigned)p.H), first = (int)(blockIdx.x / (unsigned)p.H) * 16 * kNT;
  const int kv = head / p.kv_groups, K = p.K;

  const uint16_t* w[4] = {p.w_v + ((long)head * 16 + n) * K, p.w_b + ((long)kv * 16 + n) * K, p.w_c + ((long)kv * 16 + n) * K,
                          p.w_a + (long)head * K};
  const uint16_t* x[kNT];
#pragma unroll
  for (int t = 0; t < kNT; ++t)
    x[t] = p.x + (long)min(first + 16 * t + n, p.B - 1) * p.ldx;  // tokens past the batch read its last one and store nothing

  // wavefront t finishes token tile t; the state travels with the first operands
  const int token = first + 16 * wave + n;
  const bool mine = wave < kNT && token < p.B;
  const long unit = (long)token * p.H + head;
  float4 h = make_float4(0.0f, 0.0f, 0.0f, 0.0f), c_prev = h;
  float r = 0.0f, ba = 0.0f;
  int at = 0;
  uint2 bb = make_uint2(0, 0), bc = bb;
  if (mine) {
    h = *reinterpret_cast<const float4*>(p.h + unit * 16 + 4 * q);
    c_prev = *reinterpret_cast<const float4*>(p.c_prev + unit * 16 + 4 * q);
    r = p.r[unit];
    at = p.pos[token];
    bb = *reinterpret_cast<const uint2*>(p.b_b + kv * 16 + 4 * q);
    bc = *reinterpret_cast<const uint2*>(p.b_c + kv * 16 + 4 * q);
    ba = Bf16::lo(p.b_a[head]);
  }

  f32x4_t acc[4][kNT], sum[4];
  quarter_product<kNT, kChunk>(w, x, K, wave, q, acc);
  add_quarters<kNT>(partial, acc, wave, lane, sum);
  if (!mine) return;

  const float bias_b[4] = {Bf16::lo(bb.x), Bf16::hi(bb.x), Bf16::lo(bb.y), Bf16::hi(bb.y)};
  const float bias_c[4] = {Bf16::lo(bc.x), Bf16::hi(bc.x), Bf16::lo(bc.y), Bf16::hi(bc.y)};
  const bool boundary = at == p.block_len - 1;
  const float gate = sigmoid(sum[3][0] + ba), a = gate > kCoeffFloor ? gate : 0.0f;
  const float r_new = a * r;
  float hf[4] = {h.x, h.y, h.z, h.w}, of[4];
  const float pf[4] = {c_prev.x, c_prev.y, c_prev.z, c_prev.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    hf[i] = fmaf(a, hf[i], sigmoid(sum[1][i] + bias_b[i]) * sum[0][i]);
    of[i] = fmaf(fmaf(r_new, pf[i], hf[i]), sum[2][i] + bias_c[i], sum[0][i]);
  }
  *reinterpret_cast<uint2*>(p.out + unit * 16 + 4 * q) = make_uint2(Bf16::pack2(of[0], of[1]), Bf16::pack2(of[2], of[3]));
  float4 next = make_float4(hf[0], hf[1], hf[2], hf[3]);
  if (boundary) {
    *reinterpret_cast<float4*>(p.c_prev + unit * 16 + 4 * q) = next;
    next = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
  *reinterpret_cast<float4*>(p.h + unit * 16 + 4 * q) = next;
  if (q == 0) p.r[unit] = boundary ? 1.0f : r_new;
}

template <int kNT, int kChunk>
void launch(const LayerTokenArgs& p, hipStream_t s) {
  const long tiles = (p.B + 16 * kNT - 1) / (16 * kNT);
  hipLaunchKernelGGL((layer_token_kernel<kNT, kChunk>), dim3((unsigned)(p.H * tiles)), dim3(256), 0, s, p);
}

}  // namespace

hipError_t layer_token(const LayerTokenArgs& p, hipStream_t s) {
  // Few workgroups: as many as there are. Else more tokens to a workgroup, which reads the weights less often. One / two / four
  // token tiles, us: B=32 128 heads (256 pairs) 12.5 / 14.3 / 15.2; B=256 32 heads (512) 8.8 / 7.7 / 8.9; B=1024 32 heads (2048)
  // 22.6 / 21.3 / 14.0; B=256 128 heads (2048) 65 / 48 / 32.
  const long pairs = (long)p.H * ((p.B + 15) / 16);
  const int nt = pairs <= 256 ? 1 : pairs <= 512 ? 2 : 4;
  if (nt == 1) launch<1, 4>(p, s);
  else if (nt == 2) launch<2, 4>(p, s);
  else launch<4, 2>(p, s);
  if (const hipError_t err = hipGetLastError(); err != hipSuccess) return err;
  // every wavefront of a row has to have read pos: a launch of its own (4.4 us), or with the next kernel on the stream
  return p.advance ? advance_block_positions(p.pos, p.B, p.block_len, s) : hipSuccess;
}

}  // namespace spear_btp
