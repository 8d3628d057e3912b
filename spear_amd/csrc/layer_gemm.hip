// The layer's linear projections at sizes where the matrix units are the limit, on gfx950 (MI355X): up to four of them on the same
// rows in one launch.
//
//     out_j[M, N_j] = x[M, K] w_j[N_j, K]^T + bias_j          bf16, fp32 sums, rounded once
//
// One workgroup of eight wavefronts per compute unit makes 256 x 256 tiles of the results, one after the other, in steps of 64 columns of K on
// v_mfma_f32_16x16x32_bf16 (2048 cycles of the matrix units per step). A wavefront owns 128 rows by 64 columns: 128 accumulators.
//   - Operands go from memory to LDS without registers (buffer_load ... lds, 16 bytes per lane, rows of 128 bytes): three stages of x
//     and two of the weights, 32 KiB each, all 160 KiB. x comes from memory and is asked for two steps ahead, the weights
//     come from L2 and are asked for when the stage before is free. Requests run on over the end of a tile into the next one, so
//     only the first tile waits for memory.
//   - 16-byte pieces are exchanged inside their row by the row's index ((row >> 1) & 7), on the way in by the lane that asks for them:
//     the reads of a fragment then touch every bank once (SQ_LDS_BANK_CONFLICT 0; a swizzle over 64-byte rows that ignored which
//     lanes share a cycle had one conflict per read and cost a fifth of the whole).
//   - The two wavefronts of a SIMD (wm = 0, 1) are half a phase apart, held there by the barriers: one reads fragments (12 reads)
//     while the other multiplies (32 instructions, 512 cycles), so neither needs a second set of fragment registers. Phases of
//     16 instructions gave 0.68 of the matrix units' cycles on an 8192^3 product, of 32 0.77.
//   - What lies past a row's end, the last row or the last column reads as zero: the descriptors of the buffer loads end with the tile's
//     last valid row, and the lanes whose piece lies past K ask past that end. K, M and N need no padding.
//   - Results are rounded, exchanged between lane rows (v_permlane16_swap) to 16 bytes per lane and stored while the next tile's
//     requests are under way; the waits count the stores, so the next tile doesn't wait for them before its second step.
//   - A tile with 128 columns or fewer spreads them over all wavefronts and skips half of the matrix instructions.
//   - Workgroups of one XCD take consecutive tiles of groups of four row panels by all columns: the panels of x and the weights
//     that are used at one time fit its L2.
//
// Measured, TFLOP/s, this kernel / the library's products: 131072 rows, K=512, N=512+512+512+32 950 / 775; N=512 960 / 850; K=1024
// N=1024 1180 / 1270; K=2048 N=2048+512+512+128 1310 / 1270. Without the stores of the results K=512 would run at 1150: they
// are what is left there (402 MB for 206 GFLOP). Long K is bound by the hand-over between the two groups of wavefronts and the chip's power:
// 8192^3 at 1470, where the library's kernel reaches 1630.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "btp_device.h"
#include "btp_launch.h"
#include "layer_mfma.h"
#include "layer_tile.h"

namespace spear_btp {

namespace {

constexpr int kTileRows = 256, kTileCols = 256, kStepK = 64;
constexpr int kStage = kTileRows * kStepK * 2;  // bytes of a stage of either operand
constexpr int kPanels = 4;                      // row panels of a group of tiles

struct Tile {
  int panel, job, col;  // 256 rows from 256 panel on, columns of out[job] from col on
};

__device__ __forceinline__ Tile tile_at(const LayerLinearArgs& p, int tiles_n, int id) {
  const int panels = (p.M + kTileRows - 1) / kTileRows, group = id / (kPanels * tiles_n), at = id - group * kPanels * tiles_n;
  const int in_group = min(kPanels, panels - group * kPanels);
  int n = at / in_group;
  Tile t{group * kPanels + at - n * in_group, 0, 0};
  while (n >= (p.N[t.job] + kTileCols - 1) / kTileCols) n -= (p.N[t.job++] + kTileCols - 1) / kTileCols;
  t.col = kTileCols * n;
  return t;
}

// The fragments of 32 columns: 8 row tiles of x, 4 column tiles of the weights, 2 KiB apart. The wait is part of the block: the
// registers are written when it ends.
__device__ __forceinline__ void read_fragments(uint32_t x, uint32_t w, i32x4_t (&fx)[8], i32x4_t (&fw)[4]) {
  asm volatile(
      "ds_read_b128 %8, %13\n ds_read_b128 %9, %13 offset:2048\n ds_read_b128 %10, %13 offset:4096\n ds_read_b128 %11, %13 offset:6144\n"
      "ds_read_b128 %0, %12\n ds_read_b128 %1, %12 offset:2048\n ds_read_b128 %2, %12 offset:4096\n ds_read_b128 %3, %12 offset:6144\n"
      "ds_read_b128 %4, %12 offset:8192\n ds_read_b128 %5, %12 offset:10240\n ds_read_b128 %6, %12 offset:12288\n"
      "ds_read_b128 %7, %12 offset:14336\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(fx[0]), "=&v"(fx[1]), "=&v"(fx[2]), "=&v"(fx[3]), "=&v"(fx[4]), "=&v"(fx[5]), "=&v"(fx[6]), "=&v"(fx[7]),
        "=&v"(fw[0]), "=&v"(fw[1]), "=&v"(fw[2]), "=&v"(fw[3])
      : "v"(x), "v"(w)
      : "memory");
}

// The same with a request between the reads and their wait: the address unit takes 16 cycles per request, 256 for a group's, and the
// reads of all four wavefronts 192 and their latency. One after the other they take longer than the 512 cycles in which the other group
// multiplies.
__device__ __forceinline__ void read_fragments(uint32_t x, uint32_t w, i32x4_t (&fx)[8], i32x4_t (&fw)[4], Rows& r, uint32_t to) {
  asm volatile(
      "ds_read_b128 %8, %13\n ds_read_b128 %9, %13 offset:2048\n ds_read_b128 %10, %13 offset:4096\n ds_read_b128 %11, %13 offset:6144\n"
      "ds_read_b128 %0, %12\n ds_read_b128 %1, %12 offset:2048\n ds_read_b128 %2, %12 offset:4096\n ds_read_b128 %3, %12 offset:6144\n"
      "ds_read_b128 %4, %12 offset:8192\n ds_read_b128 %5, %12 offset:10240\n ds_read_b128 %6, %12 offset:12288\n"
      "ds_read_b128 %7, %12 offset:14336\n"
      SPEAR_REQUEST4("%18", "%14", "%15", "%16", "%17", "%19", "%20")
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(fx[0]), "=&v"(fx[1]), "=&v"(fx[2]), "=&v"(fx[3]), "=&v"(fx[4]), "=&v"(fx[5]), "=&v"(fx[6]), "=&v"(fx[7]),
        "=&v"(fw[0]), "=&v"(fw[1]), "=&v"(fw[2]), "=&v"(fw[3])
      : "v"(x), "v"(w), "v"(r.at[0]), "v"(r.at[1]), "v"(r.at[2]), "v"(r.at[3]), "s"(to), "s"(r.of), "s"(r.further)
      : "memory", "m0", "scc");
  advance(r);
}

// kStreamed: results are stored with the non-temporal hint, so that L2 writes them back at once and not when the next tile's
// stores need the room. K=512: 223 against 236 us for the four projections of 131072 rows; K=1600: 192 against 184.
template <bool kStreamed>
__global__ __launch_bounds__(512) void layer_gemm_kernel(const LayerLinearArgs p, int tiles_n, int tiles) {
  __shared__ __attribute__((aligned(1024))) char lds[5 * kStage];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int n = lane & 15, q = lane >> 4, wm = wave >> 2, wn = wave & 3;
  const int K = p.K, ldx = (int)p.ldx, steps = (K + kStepK - 1) / kStepK;
  const int xcd = blockIdx.x & 7, slots = gridDim.x >> 3;
  const int last = (int)((long)tiles * (xcd + 1) / 8);
  int id = (int)((long)tiles * xcd / 8) + (int)(blockIdx.x >> 3);
  if (id >= last) return;

  // Requests: number i (0 .. 3) of wavefront w moves rows 32 w + 8 i .. + 7 of a stage, 16 bytes per lane
  const int row = 32 * wave + (lane >> 3);
  Rows rx, rw;
  rx.piece = rw.piece = ((lane & 7) ^ (lane >> 4)) * 16;  // rows 8 further have it 64 bytes across
  auto aim_x = [&](const Tile& t) {
    aim(rx, p.x + (long)t.panel * kTileRows * ldx, min(kTileRows, p.M - t.panel * kTileRows), ldx, K);
#pragma unroll
    for (int i = 0; i < 4; ++i) rx.at[i] = (row + 8 * i) * ldx * 2 + (i & 1 ? rx.piece ^ 64 : rx.piece);
  };
  auto aim_w = [&](const Tile& t) {
    const int cols = min(kTileCols, p.N[t.job] - t.col);
    aim(rw, p.w[t.job] + (long)t.col * K, cols, K, K);
    // wavefront wn has the rows 64 wn .. of a stage: the tile's columns in order, or 32 wn .. + 31 and these + 128 where there are
    // no more than 128 columns
    const int col = cols > 128 ? row : (row & 31) + (row >> 6) * 32 + (row & 32) * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) rw.at[i] = (col + 8 * i) * K * 2 + (i & 1 ? rw.piece ^ 64 : rw.piece);
  };
  const uint32_t base = lds_address(lds), x_to = base + wave * 4096, w_to = x_to + 3 * kStage;

  const uint32_t fragment = n * 128 + (q ^ (n >> 1)) * 16;
  const uint32_t x_at = base + wm * 128 * 128 + fragment, w_at = base + 3 * kStage + wn * 64 * 128 + fragment;
  f32x4_t acc[8][4];  // [row tile][column tile]; lane 16 q + n: columns 4 q .. 4 q + 3 of row n
  i32x4_t fx[8], fw[4];

  Tile cur = tile_at(p, tiles_n, id);
  aim_x(cur);
  aim_w(cur);
  request(rx, x_to); request(rw, w_to);
  end_rows(rx);
  end_rows(rw);
  request(rx, x_to + kStage); request(rw, w_to + kStage);
  wait_vm<8>();
  phase_barrier();
  if (wm == 1) phase_barrier();
  uint16_t bias_of[4][4];
  auto load_bias = [&](const Tile& t) {
    const uint16_t* bias = p.bias[t.job];
    const int N = p.N[t.job];
    const bool full = N - t.col > 128;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int c = t.col + (full ? 64 : 32) * wn + (full ? 32 : 128) * (j >> 1) + 16 * (j & 1) + 4 * q + e;
        bias_of[j][e] = bias != nullptr ? bias[min(c, N - 1)] : 0;
      }
  };
  load_bias(cur);
  int sx = 0, sw = 0;
  bool stored = false;  // 16 stores are among the requests that a wait counts
  while (true) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    const int N = p.N[cur.job], left = N - cur.col;
    const bool full = left > 128;
    const int span = full ? 64 : 32, across = full ? 32 : 128;  // first column of column tile j: span wn + across (j / 2) + 16 (j % 2)
    const bool more = id + slots < last;
    const Tile next = more ? tile_at(p, tiles_n, id + slots) : cur;  // past the last tile its first steps are asked for again, for nothing
    // The steps of an operand run on into the next tile's. That is seen to while the matrix units have work: reading is the longer part of a
    // phase.
    auto follow = [&](Rows& r, auto&& aim_at) {
      if (r.left < 2 * kStepK) {
        asm volatile("");
        if (r.left <= 0) aim_at(next);
        end_rows(r);
      }
    };
    auto multiply = [&](auto&& meanwhile) {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i][j] = mfma(fw[j], fx[i], acc[i][j]);
      meanwhile();
      if (full) {
#pragma unroll
        for (int j = 2; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < 8; ++i) acc[i][j] = mfma(fw[j], fx[i], acc[i][j]);
      }
      __builtin_amdgcn_s_setprio(0);
      phase_barrier();
    };
    int t = 0;
    do {
      // The weights of step t + 1 (the first ones of a tile have been asked for already) go where those of step t - 1 were, x of step
      // t + 2 where that of step t - 1 was: both groups of wavefronts have read them.
      if (t > 0) read_fragments(x_at + sx * kStage, w_at + sw * kStage, fx, fw, rw, w_to + (sw ^ 1) * kStage);
      else read_fragments(x_at + sx * kStage, w_at + sw * kStage, fx, fw);
      phase_barrier();
      multiply([&]() { follow(rx, aim_x); });
      read_fragments((x_at ^ 64) + sx * kStage, (w_at ^ 64) + sw * kStage, fx, fw, rx, x_to + (sx == 0 ? 2 : sx - 1) * kStage);
      // step t + 1 has landed: all but the request just made, and the stores if they came after step t + 1 was asked for
      if (stored) wait_vm<20>();
      else wait_vm<4>();
      stored = false;
      phase_barrier();
      multiply([&]() { follow(rw, aim_w); });
      sx = sx == 2 ? 0 : sx + 1;
      sw ^= 1;
    } while (++t < steps);
    request(rw, w_to + (sw ^ 1) * kStage);  // the next tile's second step, ahead of the stores

    if (p.bias[cur.job] != nullptr) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4_t add = {Bf16::lo(bias_of[j][0]), Bf16::lo(bias_of[j][1]), Bf16::lo(bias_of[j][2]), Bf16::lo(bias_of[j][3])};
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i][j] += add;
      }
    }
    load_bias(next);  // before the stores: the waits of the next tile don't count these loads
    const int rows = min(kTileRows, p.M - cur.panel * kTileRows);
    uint16_t* out = p.out[cur.job] + (long)cur.panel * kTileRows * N + cur.col;
    const auto desc = buffer_of(out, ((rows - 1) * N + min(kTileCols, left)) * 2);
    const bool wide = N % 8 == 0 && (reinterpret_cast<uintptr_t>(p.out[cur.job]) & 15u) == 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int c = span * wn + across * h + (q & 1) * 16 + (q >> 1) * 8, r = wm * 128 + n;
      const uint32_t to = c < left && (h == 0 || full) ? (uint32_t)(r * N + c) * 2 : kNowhere;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        // lane row q gets columns 8 (q >> 1) .. + 7 of column tile 2 h + (q & 1)
        const f32x4_t v0 = acc[i][2 * h], v1 = acc[i][2 * h + 1];
        const u32x2_t lo = __builtin_amdgcn_permlane16_swap(Bf16::pack2(v0[0], v0[1]), Bf16::pack2(v1[0], v1[1]), false, false);
        const u32x2_t hi = __builtin_amdgcn_permlane16_swap(Bf16::pack2(v0[2], v0[3]), Bf16::pack2(v1[2], v1[3]), false, false);
        const u32x4_t d = {lo[0], hi[0], lo[1], hi[1]};
        if (wide) {
          __builtin_amdgcn_raw_buffer_store_b128(d, desc, to + (uint32_t)(16 * i * N * 2), 0, kStreamed ? 2 : 0);
        } else if (to != kNowhere && r + 16 * i < rows) {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (c + e < left) out[(long)(r + 16 * i) * N + c + e] = (uint16_t)(d[e >> 1] >> (16 * (e & 1)));
        }
      }
    }
    if (!more) break;
    cur = next;
    id += slots;
    stored = wide;
  }
  if (wm == 0) phase_barrier();
  wait_vm<0>();  // the requests past the last tile write LDS
}

// ---- products that would not fill the chip with tiles of 256 x 256 --------------------------------------------------------------------
// 128 x 128 tiles, one to a workgroup of four wavefronts (64 x 64 each). Where there are more tiles than compute units, two stages of 64
// columns of K (64 KiB): two workgroups share a compute unit and one multiplies while the other waits. Else four stages (128 KiB), three
// of them under way. Requests, exchange of pieces, bounds and results are those above.
constexpr int kMidSide = 128, kMidStage = kMidSide * kStepK * 2;

// The fragments of 32 columns, four tiles of either operand, with a request as above.
__device__ __forceinline__ void read_fragments(uint32_t x, uint32_t w, i32x4_t (&fx)[4], i32x4_t (&fw)[4], Rows& r, uint32_t to) {
  asm volatile(
      "ds_read_b128 %4, %9\n ds_read_b128 %5, %9 offset:2048\n ds_read_b128 %6, %9 offset:4096\n ds_read_b128 %7, %9 offset:6144\n"
      "ds_read_b128 %0, %8\n ds_read_b128 %1, %8 offset:2048\n ds_read_b128 %2, %8 offset:4096\n ds_read_b128 %3, %8 offset:6144\n"
      SPEAR_REQUEST4("%14", "%10", "%11", "%12", "%13", "%15", "%16")
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(fx[0]), "=&v"(fx[1]), "=&v"(fx[2]), "=&v"(fx[3]), "=&v"(fw[0]), "=&v"(fw[1]), "=&v"(fw[2]), "=&v"(fw[3])
      : "v"(x), "v"(w), "v"(r.at[0]), "v"(r.at[1]), "v"(r.at[2]), "v"(r.at[3]), "s"(to), "s"(r.of), "s"(r.further)
      : "memory", "m0", "scc");
  advance(r);
}

// Launched with 256 threads. The bound of 512 leaves a wavefront 256 registers: given 512, the compiler keeps the sums in accumulation
// registers and copies them to and fro between matrix instructions (0.7 us per step instead of 0.45).
template <int kStages, bool kQuarters>
__global__ __launch_bounds__(512) void layer_gemm_mid_kernel(const LayerLinearArgs p, int tiles_n, int tiles) {
  __shared__ __attribute__((aligned(1024))) char lds[2 * kStages * kMidStage];  // the stages of x, then those of the weights
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int n = lane & 15, q = lane >> 4, wm = wave >> 1, wn = wave & 1;
  const int K = p.K, ldx = (int)p.ldx, steps = (K + kStepK - 1) / kStepK;
  // an XCD takes consecutive tiles, the columns of a row panel after another
  const int xcd = blockIdx.x & 7, first = (int)((long)tiles * xcd / 8), id = first + (int)(blockIdx.x >> 3);
  if (id >= (int)((long)tiles * (xcd + 1) / 8)) return;
  const int panel = id / tiles_n;
  int job = 0, col = id - panel * tiles_n;
  while (col >= (p.N[job] + kMidSide - 1) / kMidSide) col -= (p.N[job++] + kMidSide - 1) / kMidSide;
  col *= kMidSide;
  const int N = p.N[job], rows = min(kMidSide, p.M - panel * kMidSide), cols = min(kMidSide, N - col);

  const int row = 32 * wave + (lane >> 3);
  Rows rx, rw;
  rx.piece = rw.piece = ((lane & 7) ^ (lane >> 4)) * 16;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int piece = i & 1 ? rx.piece ^ 64 : rx.piece;
    rx.at[i] = (row + 8 * i) * ldx * 2 + piece;
    rw.at[i] = (row + 8 * i) * K * 2 + piece;
  }
  aim(rx, p.x + (long)panel * kMidSide * ldx, rows, ldx, K);
  aim(rw, p.w[job] + (long)col * K, cols, K, K);
  // the first tile of a panel's rows moves their positions on; read here, ahead of the requests, and written with the results
  const bool moves = p.pos != nullptr && job == 0 && col == 0 && (int)threadIdx.x < rows;
  int* const pos = p.pos + (long)panel * kMidSide + threadIdx.x;
  const int was = moves ? *pos : 0;

  const uint32_t fragment = lds_address(lds) + n * 128 + (q ^ (n >> 1)) * 16;
  const uint32_t x_at = fragment + wm * 64 * 128, w_at = fragment + kStages * kMidStage + wn * 64 * 128;
  f32x4_t acc[4][4], sum[4][4];  // kQuarters: of the quarter of K under way, and of those before it
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = sum[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  i32x4_t fx[2][4], fw[2][4];
  const uint32_t x_to = lds_address(lds) + wave * 4096, w_to = x_to + kStages * kMidStage;
#pragma unroll
  for (int t = 0; t < kStages - 1; ++t) {
    end_rows(rx);
    end_rows(rw);
    request(rx, x_to + t * kMidStage);
    request(rw, w_to + t * kMidStage);
  }
  end_rows(rx);
  end_rows(rw);
  const int share = quarter_steps(K);
  int stage = 0, left = share;  // instructions along K until the next quarter
  auto starts = [&]() {
    if (!kQuarters) return false;
    const bool first = left == 0;
    left = (first ? share : left) - 1;
    return first;
  };
  for (int t = 0; t < steps; ++t) {
    wait_vm<8 * (kStages - 2)>();  // step t has landed, the ones after it may be under way
    phase_barrier();               // in all wavefronts, and all have read step t - 1
    // Step t + kStages - 1 goes where step t - 1 was. Past the last step nothing is asked for (nowhere), so that the waits' counts hold.
    const uint32_t at = stage * kMidStage, to = (stage == 0 ? kStages - 1 : stage - 1) * kMidStage;
    read_fragments(x_at + at, w_at + at, fx[0], fw[0], rx, x_to + to);
    multiply_quarters(acc, sum, fw[0], fx[0], starts());
    read_fragments((x_at ^ 64) + at, (w_at ^ 64) + at, fx[1], fw[1], rw, w_to + to);
    multiply_quarters(acc, sum, fw[1], fx[1], starts());
    end_rows(rx);
    end_rows(rw);
    stage = stage == kStages - 1 ? 0 : stage + 1;
  }
  if (kQuarters) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] += sum[i][j];
  }

  if (const uint16_t* bias = p.bias[job]; bias != nullptr) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x4_t add;
#pragma unroll
      for (int e = 0; e < 4; ++e) add[e] = Bf16::lo(bias[min(col + 64 * wn + 16 * j + 4 * q + e, N - 1)]);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i][j] += add;
    }
  }
  uint16_t* out = p.out[job] + (long)panel * kMidSide * N + col;
  const bool wide = N % 8 == 0 && (reinterpret_cast<uintptr_t>(p.out[job]) & 15u) == 0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int c = 64 * wn + 32 * h + (q & 1) * 16 + (q >> 1) * 8;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x4_t v0 = acc[i][2 * h], v1 = acc[i][2 * h + 1];
      const u32x2_t lo = __builtin_amdgcn_permlane16_swap(Bf16::pack2(v0[0], v0[1]), Bf16::pack2(v1[0], v1[1]), false, false);
      const u32x2_t hi = __builtin_amdgcn_permlane16_swap(Bf16::pack2(v0[2], v0[3]), Bf16::pack2(v1[2], v1[3]), false, false);
      const u32x4_t d = {lo[0], hi[0], lo[1], hi[1]};
      const int r = 64 * wm + 16 * i + n;
      if (r >= rows || c >= cols) continue;
      uint16_t* const to = out + (long)r * N + c;
      if (wide) {
        *reinterpret_cast<u32x4_t*>(to) = d;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (c + e < cols) to[e] = (uint16_t)(d[e >> 1] >> (16 * (e & 1)));
      }
    }
  }
  if (moves) *pos = was + 1 >= p.block_len ? 0 : was + 1;
  wait_vm<0>();  // the requests past the last step write LDS
}

}  // namespace

bool layer_gemm_takes(const LayerLinearArgs& p) {
  if (p.K <= kStepK || p.K % 8 != 0 || p.ldx % 8 != 0 || p.K >= 1 << 21 || p.ldx >= 1 << 21) return false;
  long tiles = 0;
  for (int j = 0; j < p.jobs; ++j) {
    if (p.N[j] >= 1 << 21) return false;
    tiles += (p.N[j] + kMidSide - 1) / kMidSide;
  }
  return tiles * ((p.M + kMidSide - 1) / kMidSide) < 1l << 28;
}

hipError_t layer_gemm(const LayerLinearArgs& p, LayerTiles size, bool quarters, hipStream_t s) {
  const int side = size == LayerTiles::kMid ? kMidSide : kTileRows;
  int tiles_n = 0;
  for (int j = 0; j < p.jobs; ++j) tiles_n += (p.N[j] + side - 1) / side;
  const int tiles = tiles_n * ((p.M + side - 1) / side);
  if (tiles == 0) return hipSuccess;
  if (size == LayerTiles::kMid) {
    const dim3 grid((unsigned)((tiles + 7) / 8 * 8)), block(256);
    auto* const kernel = tiles <= 256 ? (quarters ? layer_gemm_mid_kernel<4, true> : layer_gemm_mid_kernel<4, false>)
                                      : (quarters ? layer_gemm_mid_kernel<2, true> : layer_gemm_mid_kernel<2, false>);
    hipLaunchKernelGGL(kernel, grid, block, 0, s, p, tiles_n, tiles);
    return hipGetLastError();
  }
  const dim3 grid(256), block(512);  // a workgroup for every compute unit
  if (p.K <= 1024) hipLaunchKernelGGL(layer_gemm_kernel<true>, grid, block, 0, s, p, tiles_n, tiles);
  else hipLaunchKernelGGL(layer_gemm_kernel<false>, grid, block, 0, s, p, tiles_n, tiles);
  return hipGetLastError();
}

}  // namespace spear_btp
