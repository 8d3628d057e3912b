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
// Many tokens go through tiles in LDS (below): there the chain of loads from L2 and their number bound the kernel above.
//
// Measured in a HIP graph, us, here / four library products and the step kernel: B=1 8 heads 4.0 / 23.8, B=1 128 heads 9.3 / 30.1, B=256
// 32 heads 5.9 / 25.7, B=1024 32 heads 8.2 / 25.8 (1.7 GFLOP; 11.8 without the tiles), B=1024 64 heads 20 / 43, 128 heads 60 / 64. The
// caller takes the library from B H K > 3 2^26 on, with kv heads shared and more than 2048 tokens from 2^26 on. The whole step as a call at
// B=1024, 32 heads: 122 us as products and a step.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "btp_device.h"
#include "btp_launch.h"
#include "layer_mfma.h"
#include "layer_tile.h"

namespace spear_btp {

namespace {

__device__ __forceinline__ float sigmoid(float z) { return __builtin_amdgcn_rcpf(1.0f + __expf(-z)); }

// The mixing stage's step for features 4 q .. 4 q + 3 of `head` of a token, with `sum` the products of v, b, c and a, on state and biases
// that the lane has loaded.
struct TokenState {
  float4 h, c_prev;
  float r, ba;
  int at;
  uint2 bb, bc;
};

__device__ __forceinline__ TokenState load_token(const LayerTokenArgs& p, int token, int head, int kv, int q) {
  const long unit = (long)token * p.H + head;
  return {*reinterpret_cast<const float4*>(p.h + unit * 16 + 4 * q), *reinterpret_cast<const float4*>(p.c_prev + unit * 16 + 4 * q),
          p.r[unit], Bf16::lo(p.b_a[head]), p.pos[token], *reinterpret_cast<const uint2*>(p.b_b + kv * 16 + 4 * q),
          *reinterpret_cast<const uint2*>(p.b_c + kv * 16 + 4 * q)};
}

__device__ __forceinline__ void step_token(const LayerTokenArgs& p, int token, int head, int q, const f32x4_t (&sum)[4], const TokenState& s) {
  const long unit = (long)token * p.H + head;
  const float bias_b[4] = {Bf16::lo(s.bb.x), Bf16::hi(s.bb.x), Bf16::lo(s.bb.y), Bf16::hi(s.bb.y)};
  const float bias_c[4] = {Bf16::lo(s.bc.x), Bf16::hi(s.bc.x), Bf16::lo(s.bc.y), Bf16::hi(s.bc.y)};
  const bool boundary = s.at == p.block_len - 1;
  const float gate = sigmoid(sum[3][0] + s.ba), a = gate > kCoeffFloor ? gate : 0.0f;
  const float r_new = a * s.r;
  float hf[4] = {s.h.x, s.h.y, s.h.z, s.h.w}, of[4];
  const float pf[4] = {s.c_prev.x, s.c_prev.y, s.c_prev.z, s.c_prev.w};
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
  TokenState state{};
  if (mine) state = load_token(p, token, head, kv, q);

  f32x4_t acc[4][kNT], sum[4];
  quarter_product<kNT, kChunk, 4>(w, x, K, wave, q, acc);
  add_quarters<kNT, 4>(partial, acc, wave, lane, sum);
  if (mine) step_token(p, token, head, q, sum, state);
}

// ---- many tokens ----------------------------------------------------------------------------------------------------------------------
// Two heads and 64 tokens to a workgroup, operands through LDS (layer_tile.h): four stages of 64 columns, the tokens' rows and of every
// matrix the two heads' 16 rows (of W_a the head's row sixteen times). Wavefront w asks for matrix w's rows and a quarter of the tokens';
// it multiplies head w & 1 with tokens 32 (w >> 1) .. + 31, so that v, b, c and a of a (feature, token) pair meet in one lane as above.
// Each workgroup reads its weights once for 64 tokens and its tokens once for two heads where the kernel above reads either per 64 by
// one, without the latency of every load in the chain.
constexpr int kTokenStages = 4, kTokenRows = 64, kTokenX = kTokenRows * 128, kTokenW = 128 * 128;  // bytes of a stage

// The fragments of 32 columns: two token tiles, one tile of each matrix; between the reads and their wait the requests of a part of a step.
__device__ __forceinline__ void read_token_fragments(uint32_t x, uint32_t w, i32x4_t (&fx)[2], i32x4_t (&fw)[4], Rows& r, uint32_t to) {
  asm volatile(
      "ds_read_b128 %2, %7\n ds_read_b128 %3, %7 offset:4096\n ds_read_b128 %4, %7 offset:8192\n ds_read_b128 %5, %7 offset:12288\n"
      "ds_read_b128 %0, %6\n ds_read_b128 %1, %6 offset:2048\n"
      SPEAR_REQUEST4("%12", "%8", "%9", "%10", "%11", "%13", "%14")
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(fx[0]), "=&v"(fx[1]), "=&v"(fw[0]), "=&v"(fw[1]), "=&v"(fw[2]), "=&v"(fw[3])
      : "v"(x), "v"(w), "v"(r.at[0]), "v"(r.at[1]), "v"(r.at[2]), "v"(r.at[3]), "s"(to), "s"(r.of), "s"(r.further)
      : "memory", "m0", "scc");
  advance(r);
}

__device__ __forceinline__ void read_token_fragments_x(uint32_t x, uint32_t w, i32x4_t (&fx)[2], i32x4_t (&fw)[4], Rows& r, uint32_t to) {
  asm volatile(
      "ds_read_b128 %2, %7\n ds_read_b128 %3, %7 offset:4096\n ds_read_b128 %4, %7 offset:8192\n ds_read_b128 %5, %7 offset:12288\n"
      "ds_read_b128 %0, %6\n ds_read_b128 %1, %6 offset:2048\n"
      SPEAR_REQUEST2("%10", "%8", "%9", "%11", "%12")
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(fx[0]), "=&v"(fx[1]), "=&v"(fw[0]), "=&v"(fw[1]), "=&v"(fw[2]), "=&v"(fw[3])
      : "v"(x), "v"(w), "v"(r.at[0]), "v"(r.at[1]), "s"(to), "s"(r.of), "s"(r.further)
      : "memory", "m0", "scc");
  advance(r);
}

// Launched with 256 threads; the bound of 512 keeps the sums out of the accumulation registers (see layer_gemm.hip).
__global__ __launch_bounds__(512) void layer_token_tile_kernel(const LayerTokenArgs p, int pairs) {
  __shared__ __attribute__((aligned(1024))) char lds[kTokenStages * (kTokenX + kTokenW)];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int n = lane & 15, q = lane >> 4, K = p.K, ldx = (int)p.ldx, steps = (K + kRowsStep - 1) / kRowsStep;
  const int pair = (int)blockIdx.x % pairs, first = (int)blockIdx.x / pairs * kTokenRows;

  Rows rx, rw;
  rx.piece = rw.piece = ((lane & 7) ^ (lane >> 4)) * 16;
  aim(rx, p.x + (long)first * ldx, min(kTokenRows, p.B - first), ldx, K);
  const uint16_t* const matrix = wave == 0 ? p.w_v : wave == 1 ? p.w_b : wave == 2 ? p.w_c : p.w_a;
  aim(rw, matrix, wave == 0 ? p.H * 16 : wave == 3 ? p.H : p.H / p.kv_groups * 16, K, K);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int piece = i & 1 ? rx.piece ^ 64 : rx.piece, head = min(2 * pair + (i >> 1), p.H - 1);
    const int of_head = wave == 3 ? head : (wave == 0 ? head : head / p.kv_groups) * 16 + 8 * (i & 1) + (lane >> 3);
    rx.at[i] = (16 * wave + 8 * (i & 1) + (lane >> 3)) * ldx * 2 + piece;  // the first two are used
    rw.at[i] = of_head * K * 2 + piece;
  }
  const int mine = 2 * pair + (wave & 1), head = min(mine, p.H - 1), kv = head / p.kv_groups;
  const uint32_t x_to = lds_address(lds) + wave * 2048, w_to = lds_address(lds) + kTokenStages * kTokenX + wave * 4096;
  const uint32_t fragment = lds_address(lds) + n * 128 + (q ^ (n >> 1)) * 16;
  const uint32_t x_at = fragment + (wave >> 1) * 4096, w_at = fragment + kTokenStages * kTokenX + (wave & 1) * 2048;
  auto request_x = [&](uint32_t to) {
    asm volatile(SPEAR_REQUEST2("%2", "%0", "%1", "%3", "%4") ::"v"(rx.at[0]), "v"(rx.at[1]), "s"(to), "s"(rx.of), "s"(rx.further)
                 : "memory", "m0", "scc");
    advance(rx);
  };
  for (int t = 0; t < kTokenStages - 1; ++t) {
    end_rows(rx);
    end_rows(rw);
    request(rw, w_to + t * kTokenW);
    request_x(x_to + t * kTokenX);
  }
  end_rows(rx);
  end_rows(rw);
  TokenState state[2] = {};  // travels with the first operands
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int token = first + 32 * (wave >> 1) + 16 * i + n;
    if (mine < p.H && token < p.B) state[i] = load_token(p, token, head, kv, q);
  }
  // [quarter of K][token tile][v, b, c, a]. Added up as the kernel above adds its wavefronts' quarters: a token's state does not depend on how
  // many others come with it, and is as far from 64 bits as there (h off by 9.2e-8 of its norm at K = 512, 1.1e-7 at 1024; in one chain over K
  // 1.4e-7 and 1.9e-7).
  f32x4_t acc[kParts][2][4];
#pragma unroll
  for (int u = 0; u < kParts; ++u)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int m = 0; m < 4; ++m) acc[u][i][m] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  i32x4_t fx[2][2], fw[2][4];
  int stage = 0, t = 0;
  auto step = [&](f32x4_t (&first)[2][4], f32x4_t (&second)[2][4]) {
    wait_vm<6 * (kTokenStages - 2)>();  // step t has landed, the ones after it may be under way
    phase_barrier();                    // in all wavefronts, and all have read step t - 1
    const int into = stage == 0 ? kTokenStages - 1 : stage - 1;  // where step t - 1 was
    const uint32_t x = x_at + stage * kTokenX, w = w_at + stage * kTokenW;
    read_token_fragments(x, w, fx[0], fw[0], rw, w_to + into * kTokenW);
    read_token_fragments_x(x ^ 64, w ^ 64, fx[1], fw[1], rx, x_to + into * kTokenX);
    multiply(first, fw[0], fx[0]);
    multiply(second, fw[1], fx[1]);
    end_rows(rx);
    end_rows(rw);
    stage = stage == kTokenStages - 1 ? 0 : stage + 1;
    ++t;
  };
#pragma unroll
  for (int u = 0; u < kParts; ++u) {
    const int end = quarter_steps(K) * (u + 1), whole = u + 1 < kParts ? min(end / 2, steps) : steps;  // a step is two instructions along K
    while (t < whole) step(acc[u], acc[u]);
    if (u + 1 < kParts && end % 2 != 0 && t < steps) step(acc[u], acc[u + 1 < kParts ? u + 1 : u]);
  }
  if (mine < p.H) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int token = first + 32 * (wave >> 1) + 16 * i + n;
#pragma unroll
      for (int u = 1; u < kParts; ++u)
#pragma unroll
        for (int m = 0; m < 4; ++m) acc[0][i][m] += acc[u][i][m];
      if (token < p.B) step_token(p, token, head, q, acc[0][i], state[i]);
    }
  }
  wait_vm<0>();  // the requests past the last step write LDS
}

template <int kNT, int kChunk>
void launch(const LayerTokenArgs& p, hipStream_t s) {
  const long tiles = (p.B + 16 * kNT - 1) / (16 * kNT);
  hipLaunchKernelGGL((layer_token_kernel<kNT, kChunk>), dim3((unsigned)(p.H * tiles)), dim3(256), 0, s, p);
}

}  // namespace

// Whether the tile kernel takes less time than four token tiles per wavefront, past 512 pairs. Both as fitted to 67 shapes (1 to 256 heads,
// 40 to 20000 tokens): tiles in rounds of 256 workgroups, longer with K; the other in proportion to its workgroups and K, a tenth more past 256 where
// four divides the heads (20 heads B=2000 14.3 / 11.7, 13 heads B=2500 8.4 / 10.3 in one chain over K). Four token tiles / the tile kernel, us: 1 head B=20000 4.0 / 7.2, 3 heads B=4096 4.3 / 5.0, 8 heads B=2048 5.7 / 5.4, B=20000 28.4 / 24.3, 9 heads B=5000 8.9 / 10.8,
// 16 heads B=1024 6.1 / 6.6, B=1500 8.0 / 6.8, 32 heads B=512 7.9 / 7.9, B=1024 11.8 / 8.2, 37 heads B=300 6.7 / 8.3, B=500 9.7 / 8.7, 64 heads
// B=200 10.8 / 10.6, B=1024 32 / 20, 128 heads B=1024 110 / 60.
static bool tiles_win(const LayerTokenArgs& p) {
  // the tile kernel's offsets are 32 bits: the largest matrix and 64 rows of tokens below 1 GiB
  if (32l * p.H * p.K >= 1l << 30 || 2l * kTokenRows * p.ldx >= 1l << 30) return false;
  // Up to 64 tokens either kernel reads each weight once, the tiles with half as many workgroups: 256 heads at K = 4096, four token tiles / the tile
  // kernel, B=33 25.9 / 31.3, B=40 27.2 / 31.2, B=48 28.6 / 28.4, B=64 31.7 / 31.8; with more heads than compute units the former has a second round.
  if (p.B <= kTokenRows && p.H <= 256) return false;
  const long row_tiles = (p.B + kTokenRows - 1) / kTokenRows, rounds = ((p.H + 1) / 2 * row_tiles + 255) / 256;
  const double tiles = 1.0 + (double)rounds * (4.2 + 0.36 * ((p.K + kRowsStep - 1) / kRowsStep));
  const long others = p.H * row_tiles;
  const double four = 3.5 + (1.6 + 0.0059 * p.K) * (double)others / 256;
  return tiles < (p.H % 4 == 0 && others > 256 ? 1.1 * four : four);
}

hipError_t layer_token(const LayerTokenArgs& p, hipStream_t s) {
  // Few workgroups: as many as there are. Else more tokens to a workgroup, which reads the weights less often, or the tile kernel where it is the
  // faster one. One / two token tiles, us: B=32 128 heads (256 pairs) 12.5 / 14.3; B=256 32 heads (512) 8.8 / 7.7.
  const long pairs = (long)p.H * ((p.B + 15) / 16);
  if (pairs <= 256) launch<1, 4>(p, s);
  else if (pairs <= 512) launch<2, 4>(p, s);
  else if (!tiles_win(p)) launch<4, 2>(p, s);
  else {
    const int head_pairs = (p.H + 1) / 2;
    hipLaunchKernelGGL(layer_token_tile_kernel, dim3((unsigned)(head_pairs * ((p.B + kTokenRows - 1) / kTokenRows))), dim3(256), 0, s, p, head_pairs);
  }
  if (const hipError_t err = hipGetLastError(); err != hipSuccess) return err;
  // every wavefront of a row has to have read pos: a launch of its own (4.4 us), or with the next kernel on the stream
  return p.advance ? advance_block_positions(p.pos, p.B, p.block_len, s) : hipSuccess;
}

}  // namespace spear_btp
