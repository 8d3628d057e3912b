// The weight gradients of a layer's projections at many tokens, on gfx950 (MI355X): up to two products over the token axis in one launch.
//
//     part_j[split, N_j, K_j] = dy_j[tokens of the split, N_j]^T x_j[tokens of the split, K_j]          bf16 in, fp32 out
//
// The results are a few hundred to a few thousand wide, the sum runs over 10^4 to 10^6 tokens: the token axis is cut into splits so that
// (splits x 256 x 256 tiles of the result) is just below a multiple of the 256 compute units, and layer_sums adds the splits and
// rounds once. The frame is that of layer_gemm.hip: one workgroup per compute unit, eight wavefronts of which one group reads fragments
// while the other multiplies, operands straight from memory to LDS ahead of their use, over the end of a unit into the next one. What differs:
//   - Both operands lie with the reduction across their rows. A step is 32 tokens by 256 columns, rows of 512 bytes; fragments come
//     out of LDS transposed (ds_read_b64_tr_b16: 16 lanes take 4 tokens by 16 columns and each gets one column's 4 tokens), twice
//     per 8 tokens. Which of the 32 tokens of an instruction is which is the same for both operands, so nothing else moves.
//   - 32-byte pieces (a fragment's 16 columns) are exchanged inside their row by a value of the token, three bits that differ over
//     the eight tokens two lane rows read at a time: no bank is asked twice.
//   - The tiles of one split are neighbours in the order of units, and an XCD takes a run of them: its workgroups go through the same
//     tokens at one time, so each is fetched about once for all tiles (720 MB from memory for 537 MB of operands and 1.8 GB of requests
//     at 131072 tokens, [1568, 512]).
//   - A split's sum is one fp32 chain over its tokens. The layer's backward asks for at least as many splits as the library's slices had, for chains
//     no longer than theirs (the same number of splits gives the library's bits): of [1568, 512] at 131072 tokens 4.6e-4 of the results are not the
//     nearest 16-bit value with 36 splits, 4.8e-4 with the library's 32 slices, 6.3e-4 with the 18 of the model alone, which
//     take as long (239 us either; [3200, 2048] in 12 in place of 7 1525 / 1492).
//   - Steps of 32 tokens, one phase each: five stages of 16 KiB for either operand, asked for four steps ahead.
//   - A unit's sums are stored as they lie in the accumulators, 1 KiB per store; only layer_sums looks at their order. A product of one
//     split (few tokens of a wide layer) is rounded and stored as it is: no fp32 array of its size is written and read (both of a layer at
//     512 tokens, dim 4096: a step of 487 us in place of 524).
//
// Measured at 131072 tokens, us with the sums, here / the library's batched product in slices and its sums: [1568, 512] 239 / 283, [512, 512]
// 81 / 90, [3136, 1024] 780 / 1041, [3200, 2048] 1525 / 1718, [2048, 2048] 854 / 935, [784, 256] 78 / 88; 65536 tokens [1813, 592] 181 / 208;
// 16384 tokens [1568, 512] 44 / 53, [512, 512] 29 / 26; one split: 512 tokens [1568, 512] 22 / 9, [6272, 2048] 28 / 24, 4096 tokens [6400, 4096]
// 213 / 240. The matrix units are busy 0.55 (K=512, at 2.7 TB/s from memory beside the
// parts) to 0.59 of the time and the chip's clock falls to 2.0 GHz: power and the reads of far tokens bound it. With the addresses of a
// step computed anew per request the same ring took 334 us at [1568, 512].
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "btp_device.h"
#include "btp_launch.h"
#include "layer_tile.h"

namespace spear_btp {

namespace {

constexpr int kSide = kWgradSide, kTokens = 32, kStages = 5;
constexpr int kStage = kTokens * kSide * 2;  // bytes of a stage of either operand

struct Unit {
  int job, n0, k0, step, steps;  // columns of dy and x from n0 / k0 on, steps of 32 tokens
  int part;                      // where its sums go
};

// The units of an XCD: a run of each job's, one job after the other, so that the XCDs share out both (their units differ in length).
struct Share {
  int first[2], count[2];
};

__device__ __forceinline__ Unit unit_at(const LayerWgradArgs& p, const Share& share, int id) {
  const int j = id >= share.count[0] ? 1 : 0;
  const LayerWgradJob& job = p.job[j];
  const unsigned u = (unsigned)(j ? share.first[1] + id - share.count[0] : share.first[0] + id);
  const unsigned tiles_n = (unsigned)(job.N + kSide - 1) / kSide, tiles = tiles_n * ((unsigned)(job.K + kSide - 1) / kSide);
  const unsigned split = u / tiles, tile = u - split * tiles, kt = tile / tiles_n;
  // the splits differ by a step at most: the first `more` have one more
  const unsigned all = (unsigned)((p.M + kTokens - 1) / kTokens), least = all / (unsigned)job.splits, more = all - least * (unsigned)job.splits;
  return {j, (int)(tile - kt * tiles_n) * kSide, (int)kt * kSide, (int)(split * least + min(split, more)), (int)(least + (split < more ? 1 : 0)),
          (int)u + (j && p.job[0].out == nullptr ? p.job[0].units : 0)};
}

// Fragments of 32 tokens: `a` .. `d` are the lane's addresses of four column tiles, 4 tokens further 2 KiB on. The waits are part of the
// blocks: the registers are written when they end.
// Between the reads and their wait two requests (SPEAR_REQUEST2): `at` are the lane's offsets, `of` the descriptor, `to` the LDS address.
__device__ __forceinline__ void read_tiles(uint32_t a, uint32_t b, uint32_t c, uint32_t d, u32x2_t (&f)[4][2], const uint32_t (&at)[2], i32x4_t of,
                                           uint32_t to) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8\n ds_read_b64_tr_b16 %1, %8 offset:2048\n ds_read_b64_tr_b16 %2, %9\n ds_read_b64_tr_b16 %3, %9 offset:2048\n"
      "ds_read_b64_tr_b16 %4, %10\n ds_read_b64_tr_b16 %5, %10 offset:2048\n ds_read_b64_tr_b16 %6, %11\n"
      "ds_read_b64_tr_b16 %7, %11 offset:2048\n"
      SPEAR_REQUEST2("%14", "%12", "%13", "%15", "0")
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(f[0][0]), "=&v"(f[0][1]), "=&v"(f[1][0]), "=&v"(f[1][1]), "=&v"(f[2][0]), "=&v"(f[2][1]), "=&v"(f[3][0]), "=&v"(f[3][1])
      : "v"(a), "v"(b), "v"(c), "v"(d), "v"(at[0]), "v"(at[1]), "s"(to), "s"(of)
      : "memory", "m0", "scc");
}

__device__ __forceinline__ void read_tiles(uint32_t a, uint32_t b, uint32_t c, uint32_t d, uint32_t a2, uint32_t b2, uint32_t c2, uint32_t d2,
                                           u32x2_t (&f)[4][2], u32x2_t (&g)[4][2], const uint32_t (&at)[2], i32x4_t of, uint32_t to) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %16\n ds_read_b64_tr_b16 %1, %16 offset:2048\n ds_read_b64_tr_b16 %2, %17\n"
      "ds_read_b64_tr_b16 %3, %17 offset:2048\n ds_read_b64_tr_b16 %4, %18\n ds_read_b64_tr_b16 %5, %18 offset:2048\n"
      "ds_read_b64_tr_b16 %6, %19\n ds_read_b64_tr_b16 %7, %19 offset:2048\n ds_read_b64_tr_b16 %8, %20\n"
      "ds_read_b64_tr_b16 %9, %20 offset:2048\n ds_read_b64_tr_b16 %10, %21\n ds_read_b64_tr_b16 %11, %21 offset:2048\n"
      "ds_read_b64_tr_b16 %12, %22\n ds_read_b64_tr_b16 %13, %22 offset:2048\n ds_read_b64_tr_b16 %14, %23\n"
      "ds_read_b64_tr_b16 %15, %23 offset:2048\n"
      SPEAR_REQUEST2("%26", "%24", "%25", "%27", "0")
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(f[0][0]), "=&v"(f[0][1]), "=&v"(f[1][0]), "=&v"(f[1][1]), "=&v"(f[2][0]), "=&v"(f[2][1]), "=&v"(f[3][0]), "=&v"(f[3][1]),
        "=&v"(g[0][0]), "=&v"(g[0][1]), "=&v"(g[1][0]), "=&v"(g[1][1]), "=&v"(g[2][0]), "=&v"(g[2][1]), "=&v"(g[3][0]), "=&v"(g[3][1])
      : "v"(a), "v"(b), "v"(c), "v"(d), "v"(a2), "v"(b2), "v"(c2), "v"(d2), "v"(at[0]), "v"(at[1]), "s"(to), "s"(of)
      : "memory", "m0", "scc");
}

__device__ __forceinline__ i32x4_t whole(const u32x2_t (&f)[2]) { return i32x4_t{(int)f[0][0], (int)f[0][1], (int)f[1][0], (int)f[1][1]}; }

__global__ __launch_bounds__(512) void layer_wgrad_kernel(const LayerWgradArgs p) {
  __shared__ __attribute__((aligned(1024))) char lds[2 * kStages * kStage];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int i16 = lane & 15, q = lane >> 4, wm = wave >> 2, wn = wave & 3;
  const int xcd = blockIdx.x & 7, slots = gridDim.x >> 3;
  Share share;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    share.first[j] = (int)((long)p.job[j].units * xcd / 8);
    share.count[j] = (int)((long)p.job[j].units * (xcd + 1) / 8) - share.first[j];
  }
  const int last = share.count[0] + share.count[1];
  int id = blockIdx.x >> 3;
  if (id >= last) return;

  // Requests: number i (0, 1) of wavefront w moves the tokens 4 w + 2 i and the next of a stage. The lane's place in a row is piece
  // (lane & 31) of 16 bytes; what belongs there is the piece whose pair is exchanged by the token's value.
  const int token = 4 * wave + (lane >> 5);
  auto piece_of = [&](int i) {
    const int t = token + 2 * i, value = (t & 3) | ((((t >> 3) ^ (t >> 4)) & 1) << 2);
    return ((lane & 31) ^ (value << 1)) * 16;
  };
  // One operand of the unit whose steps are asked for: the descriptor of its next step's rows, the lane's offsets (nowhere past the
  // operand's columns), bytes of a step, and the bytes that the operand's last step has.
  struct Side {
    i32x4_t of;
    uint32_t at[2];
    int stride, last_bytes;
  } dy, x;
  auto aim = [&](Side& s, const uint16_t* p0, int ld, int columns, int c0, int step) {
    const int width = 2 * min(kSide, columns - c0), rows = (int)((p.M - 1) % kTokens) + 1;
    s.of = words_of(p0 + (long)step * kTokens * ld + c0, (kTokens - 1) * 2 * ld + width);
    s.stride = kTokens * 2 * ld;
    s.last_bytes = (rows - 1) * 2 * ld + width;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int piece = piece_of(i);
      s.at[i] = piece < width ? (uint32_t)((token + 2 * i) * 2 * ld + piece) : kNowhere;
    }
  };
  auto advance = [&](Side& s) {
    const uint32_t low = (uint32_t)s.of[0] + (uint32_t)s.stride;
    s.of[1] += low < (uint32_t)s.stride ? 1 : 0;
    s.of[0] = (int)low;
  };
  // The next step to ask for: unit and step in it; past the last unit its steps again (for nothing, so that the counts of the waits hold).
  Unit cur = unit_at(p, share, id);
  int feed_id = id, feed_left = 0;
  bool feed_ends = false;  // the unit's last step is the operands'
  auto last_step = [&]() {
    if (feed_ends) {
      dy.of[2] = dy.last_bytes;
      x.of[2] = x.last_bytes;
    }
  };
  auto aim_at = [&](const Unit& u) {
    const LayerWgradJob& j = p.job[u.job];
    aim(dy, j.dy, j.ld_dy, j.cols_dy, u.n0, u.step);
    aim(x, j.x, j.K, j.K, u.k0, u.step);
    feed_left = u.steps;
    feed_ends = (long)(u.step + u.steps) * kTokens >= p.M;
    if (feed_left == 1) last_step();
  };
  aim_at(cur);
  const uint32_t to = lds_address(lds) + wave * 2048;
  auto next_step = [&]() {
    advance(dy);
    advance(x);
    if (--feed_left <= 1) {
      if (feed_left == 1) {
        last_step();
      } else {
        if (feed_id + slots < last) feed_id += slots;
        aim_at(unit_at(p, share, feed_id));
      }
    }
  };

  // Fragment addresses: token 8 q + (i16 >> 2) of the 32, its piece of 8 bytes i16 & 3, column tile c at piece pair c ^ value
  const int value = (i16 >> 2) | (((q ^ (q >> 1)) & 1) << 2);
  const uint32_t base = lds_address(lds) + (8 * q + (i16 >> 2)) * 512 + (i16 & 3) * 8;
  f32x4_t acc[8][4];  // [tile of dy's columns][tile of x's columns]; lane 16 q + n: x columns 4 q .. 4 q + 3 of dy column n
  u32x2_t fa[4][2], fb[4][2], fc[4][2];

  for (int i = 0; i < kStages - 1; ++i) {
    asm volatile(SPEAR_REQUEST2("%2", "%0", "%1", "%3", "0") ::"v"(dy.at[0]), "v"(dy.at[1]), "s"(to + i * kStage), "s"(dy.of) : "memory", "m0", "scc");
    asm volatile(SPEAR_REQUEST2("%2", "%0", "%1", "%3", "0")
                 ::"v"(x.at[0]), "v"(x.at[1]), "s"(to + (kStages + i) * kStage), "s"(x.of) : "memory", "m0", "scc");
    next_step();
  }
  wait_vm<12>();
  phase_barrier();
  if (wm == 1) phase_barrier();
  int stage = 0;
  int stored = 0;  // waits ahead of which the 32 stores of a unit may still be under way
  while (true) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    const LayerWgradJob& job = p.job[cur.job];
    const bool full = job.K - cur.k0 > 128;                // else wavefront wn has 32 columns of x
    const bool some = job.N - cur.n0 > 128 * wm;           // else this group has no columns of dy
    const uint32_t y_at = base + wm * 256 + value * 32;    // column tiles 8 wm + c: the low three bits are exchanged
    const int x_tile = full ? 4 * wn : 2 * wn;
    int t = 0;
    do {
      const uint32_t a = y_at + stage * kStage, c = base + (kStages + stage) * kStage;
      const uint32_t into = to + (stage == 0 ? kStages - 1 : stage - 1) * kStage;  // four steps ahead, where the step before this one was
      auto xa = [&](int j) { return c + (uint32_t)(((x_tile + j) ^ value) * 32); };
      read_tiles(xa(0), xa(1), xa(2), xa(3), a, a ^ 32, a ^ 64, a ^ 96, fc, fa, dy.at, dy.of, into);
      read_tiles(a ^ 128, a ^ 160, a ^ 192, a ^ 224, fb, x.at, x.of, into + kStages * kStage);
      // the next step has landed: all but the three after it, and the stores if those came after the next step was asked for
      if (stored > 0) wait_vm<44>();
      else wait_vm<12>();
      --stored;
      stage = stage == kStages - 1 ? 0 : stage + 1;
      phase_barrier();
      __builtin_amdgcn_s_setprio(1);
      auto multiply = [&](int j) {
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i][j] = mfma(whole(fc[j]), whole(i < 4 ? fa[i] : fb[i - 4]), acc[i][j]);
      };
      if (some) {
        multiply(0);
        multiply(1);
      }
      next_step();  // here, where the matrix units have work: reading is the longer part of a phase
      if (some && full) {
        multiply(2);
        multiply(3);
      }
      __builtin_amdgcn_s_setprio(0);
      phase_barrier();
    } while (++t < cur.steps);

    if (job.out != nullptr) {
      // The same number of stores, 8 bytes per lane: columns 4 q .. + 3 of x's tile j, row i16 of dy's tile i
      const int rows = min(kSide, job.N - cur.n0), cols = min(kSide, job.K - cur.k0);
      const auto desc = buffer_of(job.out + (long)cur.n0 * job.K + cur.k0, ((rows - 1) * job.K + cols) * 2);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int c = 16 * (x_tile + j) + 4 * q;
        const uint32_t at = c < cols && (full || j < 2) ? (uint32_t)((128 * wm + i16) * job.K + c) * 2 : kNowhere;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const u32x2_t d = {Bf16::pack2(acc[i][j][0], acc[i][j][1]), Bf16::pack2(acc[i][j][2], acc[i][j][3])};
          __builtin_amdgcn_raw_buffer_store_b64(d, desc, at + (uint32_t)(16 * i * job.K * 2), 0, 0);
        }
      }
    } else {
      float* const part = p.parts + ((long)cur.part * 8 + wave) * (8 * 4 * 64 * 4) + lane * 4;
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) __builtin_nontemporal_store(acc[i][j], reinterpret_cast<f32x4_t*>(part + (i * 4 + j) * 256));
    }
    if (id + slots >= last) break;
    id += slots;
    cur = unit_at(p, share, id);
    stored = 3;
  }
  if (wm == 0) phase_barrier();
  wait_vm<0>();  // the requests past the last unit write LDS
}

}  // namespace

hipError_t layer_wgrad(const LayerWgradArgs& p, hipStream_t s) {
  if (p.job[0].units + p.job[1].units == 0) return hipSuccess;
  hipLaunchKernelGGL(layer_wgrad_kernel, dim3(256), dim3(512), 0, s, p);
  return hipGetLastError();
}

int layer_wgrad_splits(long M, int N, int K, int atleast) {
  const long steps = (M + kTokens - 1) / kTokens, tiles = (long)((N + kSide - 1) / kSide) * ((K + kSide - 1) / kSide);
  const int from = (int)std::max(1l, std::min({(long)atleast, 256l, steps}));
  int best = from;
  double least = 0.0;
  for (int n = from; n <= 256 && (n == from || steps >= 16l * n); ++n) {
    // rounds of the chip, a step 0.75 us and 4 us to start and store; the sums 256 KiB per unit written and read at 4.5 TB/s
    const double us = (double)((tiles * n + 255) / 256) * (0.75 * (double)((steps + n - 1) / n) + 4.0) + 0.117 * (double)(tiles * n);
    if (n == from || us < least) {
      least = us;
      best = n;
    }
  }
  return best;
}

}  // namespace spear_btp
