// Streaming form of the operator on gfx950: prompt prefill with the state hand-over, and the
// one-token decode step. They stand where the reference has pure PyTorch loops
//   jagged_band_infer_sequential  spear/nn/phalanx/inference.py:36-92
//   JaggedBandState.step          spear/nn/phalanx/inference.py:121-140
//   step_jagged                   spear/nn/phalanx/inference.py:178-278
//   parallel_jagged               spear/nn/phalanx/inference.py:281-360
//
// Prefill is the forward recurrence kernel (same span / lane layout, swizzled LDS images and
// halo recompute as btp_scan.hip) with three additions: the epilogue y * C + V applied in
// registers before the coalesced store, an optional carry into the first block, and the state a
// decoder continues from (block-local state, in-block gate product, previous block's terminal
// state) written by the 16 lanes that own the row's last step. Prompts have any length, so rows
// that are not 16-byte aligned are handled too, by realigning 32-bit words in registers. A second
// tile kernel covers what the first does not (fp32 tensors, other block lengths and head sizes), and a kernel of one thread per
// block the rows and blocks that are too short or too long for it.
//
// The step kernel is element-wise over [B, H, D]: a thread owns 8 consecutive channels of one head
// (one 16-byte access per 16-bit operand), the per-head scalars are read by every thread of the
// head and written by the first. State may alias (in-place update): every thread reads all it
// needs before it writes, and the threads that share a head's scalar sit in one wavefront.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "btp_device.h"
#include "btp_launch.h"
#include "btp_staging.h"

namespace spear_btp {

namespace {

// ---- run-time typed scalar access (state vectors and per-head scalars: a few values per row) ----
__device__ __forceinline__ float load_scalar(const void* p, long i, int dt) {
  if (dt == kF32) return static_cast<const float*>(p)[i];
  const uint32_t w = static_cast<const uint16_t*>(p)[i];
  return dt == kBf16 ? Bf16::lo(w) : Fp16::lo(w);
}

__device__ __forceinline__ void store_scalar(void* p, long i, int dt, float v) {
  if (dt == kF32) static_cast<float*>(p)[i] = v;
  else static_cast<uint16_t*>(p)[i] = (uint16_t)((dt == kBf16 ? Bf16::pack2(v, 0.0f) : Fp16::pack2(v, 0.0f)) & 0xffffu);
}

// Block-local state and inclusive gate product after step `upto` of the block starting at kFirst.
template <int kFirst>
__device__ __forceinline__ void local_state_at(const float (&a)[32], const float (&x)[32], int upto, float& h_at,
                                               float& r_at) {
  float h = 0.0f, r = 1.0f;
  h_at = 0.0f;
  r_at = 1.0f;
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    h = fmaf(a[kFirst + q], h, x[kFirst + q]);
    r *= a[kFirst + q];
    if (q == upto) { h_at = h; r_at = r; }
  }
}

// ==========================================================================================
// Prefill, tiled: 16-bit tensors, 16 channels, block length 16
// ==========================================================================================
// kAlign: what every channel row's start is aligned to, in bytes (1: rows alternate between a word and an odd
// element -- L odd, word-aligned tensors -- which is kRowsAlternate of the staging helpers). 16: L is a multiple of 8 and every
// pointer 16-byte aligned (16-byte accesses); 4 or 2: rows of any length (see
// slab16_global_to_regs_ragged), starting on words when L is even and the tensors are word-aligned.
template <class E, class C, bool kEpilogue, bool kStreamIn, int kAlign>
__global__ __launch_bounds__(64 * kWaves) void jagged_prefill_kernel(
    const typename C::elem* __restrict__ coeff, const uint16_t* __restrict__ x, const uint16_t* __restrict__ cmul,
    const uint16_t* __restrict__ vadd, const void* __restrict__ carry_init, uint16_t* __restrict__ y,
    void* __restrict__ h_tail, void* __restrict__ r_tail, void* __restrict__ c_prev_tail, int state_dtype,
    int r_dtype, int L, int spans_per_row, long total_spans) {
  constexpr bool kRagged = kAlign < 16;
  constexpr int kRows = kAlign == 4 ? kRowsOnWords : kAlign == 1 ? kRowsAlternate : kRowsAnywhere;
  constexpr int kImages = kEpilogue ? 3 : 1;
  __shared__ __align__(16) unsigned char lds[kWaves][kImages * 4096 + kCoeffLdsBytes];

  // rows of several spans: the carry into a span's first block comes from the neighbouring
  // wavefront through LDS (one workgroup barrier), as in the forward kernel
  constexpr bool kHandOver = !kStreamIn && kWaves > 1;
  __shared__ float left_state[kHandOver ? kWaves : 1][kChan];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const long span = first_span_of_workgroup<(SPEAR_BTP_XCD_REMAP == 2) || (SPEAR_BTP_XCD_REMAP == 1 && !kStreamIn)>() + wave;
  if (span >= total_spans) {  // wave-uniform
    if constexpr (kHandOver) __syncthreads();  // keep the barrier count equal for every wavefront
    return;
  }
  const SpanCoord sc = span_coord(span, spans_per_row, L);

  unsigned char* img = lds[wave];
  float* a_lds = reinterpret_cast<float*>(img + kImages * 4096);
  const long slab_off = (sc.row * kChan) * (long)L + sc.s0;
  const typename C::elem* arow = coeff + sc.row * (long)L + sc.s0;
  const int j = lane >> 4, d = lane & 15;

  uint4 xin[4], cin[4], vin[4];
  uint32_t xw[kRagged ? 16 : 1], cw[kRagged ? 16 : 1], vw[kRagged ? 16 : 1];  // the ragged path's words
  uint32_t xe = 0u, ce = 0u, ve = 0u;
  typename C::pair_t ain;
  if constexpr (kRagged) {
    slab16_global_to_regs_ragged<kRows>(x + slab_off, L, sc.nvalid, lane, xw, xe);
    ain = coeff_global_to_reg_ragged<C>(arow, sc.nvalid, lane);
    if constexpr (kEpilogue) {
      slab16_global_to_regs_ragged<kRows>(cmul + slab_off, L, sc.nvalid, lane, cw, ce);
      slab16_global_to_regs_ragged<kRows>(vadd + slab_off, L, sc.nvalid, lane, vw, ve);
    }
  } else {
    slab16_global_to_regs<nt_loads(kStreamIn)>(x + slab_off, L, sc.nvalid, lane, xin);
    ain = coeff_global_to_reg<C>(arow, sc.nvalid, lane);
    if constexpr (kEpilogue) {
      slab16_global_to_regs<true>(cmul + slab_off, L, sc.nvalid, lane, cin);  // read once, by this span only
      slab16_global_to_regs<true>(vadd + slab_off, L, sc.nvalid, lane, vin);
    }
  }

  float c_halo = 0.0f;
  if (j == 0) {
    if (sc.sp > 0 && !(kHandOver && wave > 0)) {  // local terminal state of the block left of the span, channel d
      float ah[16], xh[16];
      const uint16_t* xp = x + slab_off + (long)d * L - kTile;
      if constexpr (kRagged) {
        C::load_block_ragged(arow - kTile, ah);
        unpack8<E>(load16_plain_unaligned(xp), xh);
        unpack8<E>(load16_plain_unaligned(xp + 8), xh + 8);
      } else {
        C::load_block(arow - kTile, ah);
        unpack8<E>(*reinterpret_cast<const uint4*>(xp), xh);
        unpack8<E>(*reinterpret_cast<const uint4*>(xp + 8), xh + 8);
      }
      float h = 0.0f;
#pragma unroll
      for (int r = 0; r < 16; ++r) h = fmaf(ah[r], h, xh[r]);
      c_halo = h;
    } else if (sc.sp == 0 && carry_init != nullptr) {
      c_halo = load_scalar(carry_init, sc.row * kChan + d, state_dtype);
    }
  }

  coeff_reg_to_lds<C>(a_lds, lane, ain);
  if constexpr (kRagged) {
    slab16_regs_realign<kRows>(x + slab_off, L, sc.nvalid, lane, xw, xe);
    slab16_regs_to_lds_ragged(img, lane, xw);
    if constexpr (kEpilogue) {
      slab16_regs_realign<kRows>(cmul + slab_off, L, sc.nvalid, lane, cw, ce);
      slab16_regs_to_lds_ragged(img + 4096, lane, cw);
      slab16_regs_realign<kRows>(vadd + slab_off, L, sc.nvalid, lane, vw, ve);
      slab16_regs_to_lds_ragged(img + 8192, lane, vw);
    }
  } else {
    slab16_regs_to_lds(img, lane, xin);
    if constexpr (kEpilogue) {
      slab16_regs_to_lds(img + 4096, lane, cin);
      slab16_regs_to_lds(img + 8192, lane, vin);
    }
  }
  wave_lds_handover();

  float xf[32], a[32], yv[32];
  lane_read16<E>(img, j, d, xf);
  coeff_lane_read(a_lds, j, a);

  // Same three chains as the forward kernel: local run through block A, continued into block B
  // (B's outputs); B's own local terminal state for the next lane group; A from its carry.
  float h = 0.0f;
#pragma unroll
  for (int r = 0; r < 16; ++r) h = fmaf(a[r], h, xf[r]);
  const float vA_last = h;
#pragma unroll
  for (int r = 16; r < 32; ++r) {
    h = fmaf(a[r], h, xf[r]);
    yv[r] = h;
  }
  float vB_last = 0.0f;
#pragma unroll
  for (int r = 16; r < 32; ++r) vB_last = fmaf(a[r], vB_last, xf[r]);
  const float from_left = lane_rotate(vB_last, lane, -16);
  if constexpr (kHandOver) {
    if (j == 3) left_state[wave][d] = vB_last;
    __syncthreads();
    if (sc.sp > 0 && wave > 0 && j == 0) c_halo = left_state[wave - 1][d];
  }
  const float cA = j == 0 ? c_halo : from_left;
  h = cA;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    h = fmaf(a[r], h, xf[r]);
    yv[r] = h;
  }

  // ---- hand-over state, by the lanes that own the row's last step (wave-uniform conditions)
  if (h_tail != nullptr && sc.sp == spans_per_row - 1) {
    const int p = sc.nvalid - 1, q = p & 31;
    if (j == (p >> 5)) {
      const bool in_b = q >= 16;  // the last step lies in the lane's second block
      float ht, rt;
      // two copies with constant indices: selecting between array elements at run time would
      // move the register arrays to scratch memory
      if (in_b) local_state_at<16>(a, xf, q & 15, ht, rt);
      else local_state_at<0>(a, xf, q & 15, ht, rt);
      const bool full = (q & 15) == 15;
      const float prev = in_b ? vA_last : cA;  // terminal local state of the block before (0 / carry_init at the row start)
      const long o = sc.row * kChan + d;
      store_scalar(h_tail, o, state_dtype, ht);
      store_scalar(c_prev_tail, o, state_dtype, full ? ht : prev);
      if (d == 0) store_scalar(r_tail, sc.row, r_dtype, full ? 1.0f : rt);
    }
  }

  if constexpr (kEpilogue) {
    float cf[32];
    lane_read16<E>(img + 4096, j, d, cf);
#pragma unroll
    for (int r = 0; r < 32; ++r) yv[r] *= cf[r];
    lane_read16<E>(img + 8192, j, d, cf);
#pragma unroll
    for (int r = 0; r < 32; ++r) yv[r] += cf[r];
  }

  wave_lds_handover();
  lane_write16<E>(img, j, d, yv);
  wave_lds_handover();
  if constexpr (kRagged) slab16_lds_to_global_ragged<kRows>(img, y + slab_off, L, sc.nvalid, lane, sc.nvalid == L);
  else slab16_lds_to_global<true>(img, y + slab_off, L, sc.nvalid, lane);
}

// ==========================================================================================
// Element access by index, for the kernels below
// ==========================================================================================
struct F32Elt {};

template <class T>
struct Scalar;
template <>
struct Scalar<Bf16> {
  typedef uint16_t type;
  static __device__ __forceinline__ float get(const type* p, long i) { return Bf16::lo(p[i]); }
  static __device__ __forceinline__ void put(type* p, long i, float v) { p[i] = (uint16_t)(Bf16::pack2(v, 0.0f) & 0xffffu); }
};
template <>
struct Scalar<Fp16> {
  typedef uint16_t type;
  static __device__ __forceinline__ float get(const type* p, long i) { return Fp16::lo(p[i]); }
  static __device__ __forceinline__ void put(type* p, long i, float v) { p[i] = (uint16_t)(Fp16::pack2(v, 0.0f) & 0xffffu); }
};
template <>
struct Scalar<F32Elt> {
  typedef float type;
  static __device__ __forceinline__ float get(const type* p, long i) { return p[i]; }
  static __device__ __forceinline__ void put(type* p, long i, float v) { p[i] = v; }
};

// ==========================================================================================
// Prefill, any element type, head size and block length: fp32 tensors, other D / block_len, fp32 linear gates.
//
// Bound by HBM (four tensors once through). A wavefront owns a tile of 16 channel rows x `lanes` lane groups of
// `per_lane` whole blocks each, about 64 steps: lane (j, d) runs channel row d through its blocks. x is moved in memory
// order (granules of kG bytes per lane, neighbouring lanes on neighbouring granules of a row) into an fp32 image in
// LDS, where rows may start anywhere, and the recurrence's results replace it there; c and v never touch LDS, they
// are loaded in the same memory order ahead of the arithmetic and applied on the way out. The image's rows are an odd number of
// 16-byte chunks apart, so the per-channel reads hit different banks. As in the tiled kernel the carry into a tile
// comes from the wavefront before it through LDS behind one barrier, and a workgroup's first wavefront reads the
// block before its tile instead. One thread per (row, channel, block), the first form of this kernel, had every lane of
// a wavefront on a line of its own: fp32, B=64 H=32 D=16 L=1000 (532 MB) took 1412 us where this one takes 95 us.
// ==========================================================================================
constexpr int kTileRows = 16;   // channel rows of a tile
constexpr int kTileWaves = 4;   // wavefronts of a workgroup: consecutive tiles of the same channel rows
constexpr int kOutside = 0x7ffffff0;  // a byte offset past every buffer resource: loads give 0, stores are dropped

struct TileArgs {
  const void *coeff, *x, *c, *v, *carry_init;
  void *y, *h_tail, *r_tail, *c_prev_tail;
  long rd_total;     // channel rows: B * H * D
  long tensor_bytes;
  int D, L, nblk;
  int block_len;  // of the tiles: the streaming form's, or L where that is longer than the rows
  int whole;      // steps of a complete block
  int a_dtype, log_a, state_dtype, r_dtype;
  int lanes, per_lane;    // lane groups in use, blocks per lane group
  int spans;              // tiles per channel row
  long tiles;
  int main_gpr, halo_gpr;     // granules that cover a row's part of the tile, of the block before it
  uint32_t main_magic, halo_magic;  // ceil(2^20 / gpr): idx / gpr == (idx * magic) >> 20 for every index of a tile
  int stride;                 // floats between the image's rows
  int wave_floats;            // LDS of one wavefront
};

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// kG bytes of one row: 16 (rows on the 16-byte grid), 4 (on words; a 16-bit row may start on a word's second half) or
// 2 (16-bit tensors that do not even start on words, or not all on the same half).
template <class T, int kG>
struct Granule {
  static constexpr int kBytes = sizeof(typename Scalar<T>::type);
  static constexpr int kE = kG / kBytes;
  static constexpr bool kHalves = kBytes == 2 && kG == 4;  // row starts may fall inside a granule
  typedef typename std::conditional<kG == 16, u32x4_t, uint32_t>::type reg_t;

  // Streaming policy where a line is read once. 16-bit rows off the 16-byte grid share words and lines between tiles: cached loads there
  // (B=16 H=16 D=64 L=2047 bf16: 140 -> 111 us), and cached stores everywhere (a tile writes part of a line at each end of its
  // rows: B=64 H=32 L=1000 fp32 102 -> 95 us).
  static __device__ __forceinline__ reg_t load(__amdgpu_buffer_rsrc_t r, int off) {
    if constexpr (kG == 16) return __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 2);
    else if constexpr (kBytes == 4) return __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 2);
    else if constexpr (kG == 4) return __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
    else return __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0);
  }
  static __device__ __forceinline__ void unpack(const reg_t& g, float (&f)[kE]) {
    if constexpr (kG == 16) {
#pragma unroll
      for (int i = 0; i < kE; ++i) {
        if constexpr (kBytes == 4) f[i] = __uint_as_float(g[i]);
        else f[i] = (i & 1) ? T::hi(g[i >> 1]) : T::lo(g[i >> 1]);
      }
    } else if constexpr (kBytes == 4) {
      f[0] = __uint_as_float(g);
    } else {
      f[0] = T::lo(g);
      if constexpr (kE == 2) f[1] = T::hi(g);
    }
  }
};

// Where one lane's granule of a tile lies: byte offset from the tile's base, and the columns (steps) it covers.
struct GranuleAt {
  int row, col, off;
  bool live;
};

// kN: granules per lane that cover a tile of 64 steps; larger tiles (blocks above 64 steps) take several rounds.
template <class T, int kG, int kN, bool kShared, int kBL>
__global__ __launch_bounds__(64 * kTileWaves) void jagged_prefill_tile_kernel(const TileArgs p) {
  typedef Granule<T, kG> G;
  constexpr int kE = G::kE, kBytes = G::kBytes;
  extern __shared__ __align__(16) float tile_lds[];
  __shared__ float left_state[kTileWaves][kTileRows];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int j = lane >> 4, d = lane & 15;
  const long tile = first_span_of_workgroup<true>(kTileWaves) + wave;
  if (tile >= p.tiles) {  // wave-uniform
    __syncthreads();
    return;
  }
  const int bl = kBL ? kBL : p.block_len;
  const int per_lane = kBL ? 1 : p.per_lane, lanes = kBL ? 4 : p.lanes;
  const int L = p.L;
  const long group = tile / p.spans;
  const int sp = (int)(tile - group * p.spans);
  const long rd0 = group * kTileRows;
  const int rows = (int)min((long)kTileRows, p.rd_total - rd0);
  const int i0 = sp * lanes * per_lane;          // first block of the tile
  const int s0 = i0 * bl, W = lanes * per_lane * bl;
  const int n = min(W, L - s0);                  // steps of the tile that exist
  const bool last = sp == p.spans - 1;
  const bool halo = sp > 0 && wave == 0;         // the block before the tile is read here

  float* img = tile_lds + wave * p.wave_floats;  // columns [pad - bl, pad): the block before; [pad, pad + W): the tile
  const int pad = (bl + 3) & ~3;
  float* a_lds = img + kTileRows * p.stride;     // gates, same columns as the image
  const int stride = p.stride;

  // A tile's base is moved to the granule that holds its first element (kHalves), so granule offsets stay aligned.
  auto base_of = [&](int s) {
    long e = rd0 * (long)L + s;
    return G::kHalves ? (e & ~1L) : e;
  };
  auto rsrc = [&](const void* q, int s) {
    const long b = base_of(s) * kBytes;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(static_cast<const char*>(q) + b), 0,
                                             (int)min(p.tensor_bytes - b, 0x70000000L), 0x00020000);
  };
  auto place = [&](int idx, int s, int gpr, uint32_t magic, int width) {
    GranuleAt g;
    g.row = (int)(((uint32_t)idx * magic) >> 20);
    const int k = idx - g.row * gpr;
    int e = g.row * L;
    int shift = 0;
    if constexpr (G::kHalves) {
      e += (int)((rd0 * (long)L + s) & 1);
      shift = e & 1;
      e -= shift;
    }
    g.col = k * kE - shift;
    g.live = g.row < rows && g.col < width;
    g.off = g.live ? (e + k * kE) * kBytes : kOutside;
    return g;
  };
  // The tensor's last word when only its first half exists: the word load above is out of bounds there.
  const bool half_end = G::kHalves && (p.rd_total * (long)L) % 2 != 0 && last && rd0 + rows == p.rd_total;
  auto reload_half = [&](typename G::reg_t& w, __amdgpu_buffer_rsrc_t r, const GranuleAt& g, int s) {
    if constexpr (G::kHalves) {
      if (half_end && g.live && base_of(s) * kBytes + g.off + 4 > p.tensor_bytes) w = __builtin_amdgcn_raw_buffer_load_b16(r, g.off, 0, 0);
    }
  };
  auto to_image = [&](const typename G::reg_t& w, const GranuleAt& g, int col0, int width) {
    float f[kE];
    G::unpack(w, f);
    float* dst = img + g.row * stride + col0 + g.col;
    if constexpr (kG == 16) {
      if (g.live) {
#pragma unroll
        for (int q = 0; q < kE; q += 4) *reinterpret_cast<float4*>(dst + q) = make_float4(f[q], f[q + 1], f[q + 2], f[q + 3]);
      }
    } else {
      if (g.live && g.col >= 0) dst[0] = f[0];
      if constexpr (kE == 2) {
        if (g.live && g.col + 1 < width) dst[1] = f[1];
      }
    }
  };

  // ---- every global read of the first round, before anything waits
  const __amdgpu_buffer_rsrc_t rx = rsrc(p.x, s0);
  const bool epilogue = p.c != nullptr;
  typename G::reg_t xin[kN], cin[kN], vin[kN];
#pragma unroll
  for (int i = 0; i < kN; ++i) xin[i] = G::load(rx, place(64 * i + lane, s0, p.main_gpr, p.main_magic, n).off);
  const __amdgpu_buffer_rsrc_t rc = rsrc(epilogue ? p.c : p.x, s0), rv = rsrc(epilogue ? p.v : p.x, s0);
  if (epilogue) {
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const int off = place(64 * i + lane, s0, p.main_gpr, p.main_magic, n).off;
      cin[i] = G::load(rc, off);
      vin[i] = G::load(rv, off);
    }
  }
  const long row0 = rd0 / p.D;  // kShared: the one gate row of the tile's channel rows
  auto gate_at = [&](long row, int t) {
    const float g = load_scalar(p.coeff, row * (long)L + t, p.a_dtype);
    return p.log_a ? __expf(g) : g;
  };
  if constexpr (kShared) {
    for (int q = lane; q < n; q += 64) a_lds[pad + q] = gate_at(row0, s0 + q);
    if (halo)
      for (int q = lane; q < bl; q += 64) a_lds[pad - bl + q] = gate_at(row0, s0 - bl + q);
  }
  if (halo) {
    const int sh = s0 - bl;
    const __amdgpu_buffer_rsrc_t rh = rsrc(p.x, sh);
    for (int base = 0; base < kTileRows * p.halo_gpr; base += 64) {
      const GranuleAt g = place(base + lane, sh, p.halo_gpr, p.halo_magic, bl);
      typename G::reg_t w = G::load(rh, g.off);
      to_image(w, g, pad - bl, bl);
    }
  }
#pragma unroll
  for (int i = 0; i < kN; ++i) {
    const GranuleAt g = place(64 * i + lane, s0, p.main_gpr, p.main_magic, n);
    reload_half(xin[i], rx, g, s0);
    to_image(xin[i], g, pad, n);
  }
  const int granules = kTileRows * p.main_gpr;
  for (int base = 64 * kN; base < granules; base += 64 * kN) {  // block lengths above 64
    typename G::reg_t w[kN];
#pragma unroll
    for (int i = 0; i < kN; ++i) w[i] = G::load(rx, place(base + 64 * i + lane, s0, p.main_gpr, p.main_magic, n).off);
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const GranuleAt g = place(base + 64 * i + lane, s0, p.main_gpr, p.main_magic, n);
      reload_half(w[i], rx, g, s0);
      to_image(w[i], g, pad, n);
    }
  }
  wave_lds_handover();

  // ---- the recurrences, lane (j, d): channel row d, blocks i0 + j per_lane ...
  const bool worker = j < lanes;
  float* xr = img + d * stride;
  const long row_d = kShared ? row0 : min(rd0 + d, p.rd_total - 1) / p.D;
  // f(step's column, gate, x) over the block that starts at column `col`; rows and blocks past the end read columns
  // that were not written, which reach nothing that is stored
  auto over_block = [&](int col, int len, auto f) {
    if constexpr (kShared && kBL != 0) {
#pragma unroll
      for (int q = 0; q < kBL; q += 4) {
        const float4 a4 = *reinterpret_cast<const float4*>(a_lds + col + q), x4 = *reinterpret_cast<const float4*>(xr + col + q);
        f(col + q, a4.x, x4.x); f(col + q + 1, a4.y, x4.y); f(col + q + 2, a4.z, x4.z); f(col + q + 3, a4.w, x4.w);
      }
    } else {
      int q = 0;
      if constexpr (kShared) {
        if (((col | len) & 3) == 0) {
#pragma unroll 2
          for (; q < len; q += 4) {
            const float4 a4 = *reinterpret_cast<const float4*>(a_lds + col + q), x4 = *reinterpret_cast<const float4*>(xr + col + q);
            f(col + q, a4.x, x4.x); f(col + q + 1, a4.y, x4.y); f(col + q + 2, a4.z, x4.z); f(col + q + 3, a4.w, x4.w);
          }
        }
      }
      for (; q < len; ++q) {
        float a;
        if constexpr (kShared) a = a_lds[col + q];
        else a = gate_at(row_d, min(max(s0 + col + q - pad, 0), L - 1));
        f(col + q, a, xr[col + q]);
      }
    }
  };
  auto terminal = [&](int col) {
    float h = 0.0f;
    over_block(col, bl, [&](int, float a, float x) { h = fmaf(a, h, x); });
    return h;
  };
  const int col0 = pad + j * per_lane * bl;  // this lane's first column
  float from_halo = 0.0f;
  if (halo && j == 0) from_halo = terminal(pad - bl);
  float end_state = 0.0f;  // terminal local state of this lane's last block
  if (worker) end_state = terminal(col0 + (per_lane - 1) * bl);
  const float from_left = lane_rotate(end_state, lane, -16);
  if (j == lanes - 1) left_state[wave][d] = end_state;
  __syncthreads();
  float carry = from_left;
  if (j == 0) {
    carry = sp == 0 ? 0.0f : wave > 0 ? left_state[wave - 1][d] : from_halo;
    if (sp == 0 && p.carry_init != nullptr && d < rows) carry = load_scalar(p.carry_init, rd0 + d, p.state_dtype);
  }

  // ---- hand-over state, by the lanes that own the row's last block (before the image is overwritten)
  if (p.h_tail != nullptr && last) {
    const int b = p.nblk - 1 - i0 - j * per_lane;  // the last block, counted from this lane's first
    if (worker && b >= 0 && b < per_lane && d < rows) {
      const float prev = b > 0 ? terminal(col0 + (b - 1) * bl) : carry;
      const int len = L - (p.nblk - 1) * bl;
      float h = 0.0f, r = 1.0f;
      for (int q = 0; q < len; ++q) {
        const int col = col0 + b * bl + q;
        const float a = kShared ? a_lds[col] : gate_at(row_d, s0 + col - pad);
        h = fmaf(a, h, xr[col]);
        r *= a;
      }
      const long o = rd0 + d;
      store_scalar(p.h_tail, o, p.state_dtype, h);
      store_scalar(p.c_prev_tail, o, p.state_dtype, len == p.whole ? h : prev);
      if (o % p.D == 0) store_scalar(p.r_tail, o / p.D, p.r_dtype, len == p.whole ? 1.0f : r);
    }
  }

  if (worker) {
    for (int b = 0; b < per_lane; ++b) {
      float hl = 0.0f, hc = carry;
      over_block(col0 + b * bl, bl, [&](int col, float a, float x) {
        hl = fmaf(a, hl, x);
        hc = fmaf(a, hc, x);
        xr[col] = hc;
      });
      carry = hl;
    }
  }
  wave_lds_handover();

  // ---- out, in memory order
  const __amdgpu_buffer_rsrc_t ry = rsrc(p.y, s0);
  auto finish = [&](const GranuleAt& g, const typename G::reg_t& cw, const typename G::reg_t& vw) {
    if (!g.live) return;
    float f[kE];
    const float* src = img + g.row * stride + pad + g.col;
    if constexpr (kG == 16) {
#pragma unroll
      for (int q = 0; q < kE; q += 4) {
        const float4 t = *reinterpret_cast<const float4*>(src + q);
        f[q] = t.x; f[q + 1] = t.y; f[q + 2] = t.z; f[q + 3] = t.w;
      }
    } else {
#pragma unroll
      for (int q = 0; q < kE; ++q) f[q] = src[q];
    }
    if (epilogue) {
      float cf[kE], vf[kE];
      G::unpack(cw, cf);
      G::unpack(vw, vf);
#pragma unroll
      for (int q = 0; q < kE; ++q) f[q] = fmaf(f[q], cf[q], vf[q]);
    }
    if constexpr (kBytes == 4) {
      if constexpr (kG == 16) {
        const u32x4_t w = {__float_as_uint(f[0]), __float_as_uint(f[1]), __float_as_uint(f[2]), __float_as_uint(f[3])};
        __builtin_amdgcn_raw_buffer_store_b128(w, ry, g.off, 0, 0);
      } else {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(f[0]), ry, g.off, 0, 0);
      }
    } else if constexpr (kG == 16) {
      const u32x4_t w = {T::pack2(f[0], f[1]), T::pack2(f[2], f[3]), T::pack2(f[4], f[5]), T::pack2(f[6], f[7])};
      __builtin_amdgcn_raw_buffer_store_b128(w, ry, g.off, 0, 0);
    } else if constexpr (kG == 4) {
      const uint32_t w = T::pack2(f[0], f[1]);
      const bool lo = g.col >= 0, hi = g.col + 1 < n;  // which halves are this row's
      if (lo && hi) __builtin_amdgcn_raw_buffer_store_b32(w, ry, g.off, 0, 0);
      else if (lo) __builtin_amdgcn_raw_buffer_store_b16((unsigned short)(w & 0xffffu), ry, g.off, 0, 0);
      else __builtin_amdgcn_raw_buffer_store_b16((unsigned short)(w >> 16), ry, g.off + 2, 0, 0);
    } else {
      __builtin_amdgcn_raw_buffer_store_b16((unsigned short)(T::pack2(f[0], 0.0f) & 0xffffu), ry, g.off, 0, 0);
    }
  };
#pragma unroll
  for (int i = 0; i < kN; ++i) {
    const GranuleAt g = place(64 * i + lane, s0, p.main_gpr, p.main_magic, n);
    if (epilogue) {
      reload_half(cin[i], rc, g, s0);
      reload_half(vin[i], rv, g, s0);
    }
    finish(g, cin[i], vin[i]);
  }
  for (int base = 64 * kN; base < granules; base += 64 * kN) {
    typename G::reg_t cw[kN], vw[kN];
    if (epilogue) {
#pragma unroll
      for (int i = 0; i < kN; ++i) {
        const int off = place(base + 64 * i + lane, s0, p.main_gpr, p.main_magic, n).off;
        cw[i] = G::load(rc, off);
        vw[i] = G::load(rv, off);
      }
    }
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const GranuleAt g = place(base + 64 * i + lane, s0, p.main_gpr, p.main_magic, n);
      if (epilogue) {
        reload_half(cw[i], rc, g, s0);
        reload_half(vw[i], rv, g, s0);
      }
      finish(g, cw[i], vw[i]);
    }
  }
}

// ==========================================================================================
// Prefill, element-granular: rows and blocks of few steps (tiles_pay_off), blocks too long for a tile in LDS (above
// kMaxTileBlock), or rows too long for the tile kernel's 32-bit offsets. One thread per (row, channel, block); lanes run over blocks.
// ==========================================================================================
template <class T>
__global__ __launch_bounds__(256) void jagged_prefill_any_kernel(
    const void* __restrict__ coeff, int a_dtype, int log_a, const typename Scalar<T>::type* __restrict__ x,
    const typename Scalar<T>::type* __restrict__ cmul, const typename Scalar<T>::type* __restrict__ vadd,
    const void* __restrict__ carry_init, typename Scalar<T>::type* __restrict__ y, void* __restrict__ h_tail,
    void* __restrict__ r_tail, void* __restrict__ c_prev_tail, int state_dtype, int r_dtype, long rows, int D, int L,
    int block_len, int nblk) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= rows * D * nblk) return;
  const int i = (int)(idx % nblk);
  const long rd = idx / nblk;
  const int d = (int)(rd % D);
  const long row = rd / D;
  const long xo = rd * (long)L, ao = row * (long)L;

  auto gate = [&](int t) {
    const float g = load_scalar(coeff, ao + t, a_dtype);
    return log_a ? __expf(g) : g;
  };

  float carry = 0.0f;
  if (i > 0) {  // terminal local state of the block before
    for (int t = (i - 1) * block_len; t < i * block_len; ++t) carry = fmaf(gate(t), carry, Scalar<T>::get(x, xo + t));
  } else if (carry_init != nullptr) {
    carry = load_scalar(carry_init, rd, state_dtype);
  }

  const int t0 = i * block_len, t1 = min(L, t0 + block_len);
  float hl = 0.0f, hc = carry, rp = 1.0f;
  for (int t = t0; t < t1; ++t) {
    const float a = gate(t), xv = Scalar<T>::get(x, xo + t);
    hl = fmaf(a, hl, xv);
    hc = fmaf(a, hc, xv);
    rp *= a;
    float out = hc;
    if (cmul != nullptr) out = fmaf(out, Scalar<T>::get(cmul, xo + t), Scalar<T>::get(vadd, xo + t));
    Scalar<T>::put(y, xo + t, out);
  }
  if (h_tail != nullptr && i == nblk - 1) {
    const bool full = (t1 - t0) == block_len;
    store_scalar(h_tail, rd, state_dtype, hl);
    store_scalar(c_prev_tail, rd, state_dtype, full ? hl : carry);
    if (d == 0) store_scalar(r_tail, row, r_dtype, full ? 1.0f : rp);
  }
}

// ==========================================================================================
// Decode step
// ==========================================================================================
template <class T>
struct Oct;  // 8 consecutive elements
template <class E16>
struct Oct16 {
  typedef uint16_t type;
  static __device__ __forceinline__ void get(const type* p, long i, float (&v)[8]) {
    unpack8<E16>(*reinterpret_cast<const uint4*>(p + i), v);
  }
  static __device__ __forceinline__ void put(type* p, long i, const float (&v)[8]) {
    *reinterpret_cast<uint4*>(p + i) = pack8<E16>(v);
  }
};
template <>
struct Oct<Bf16> : Oct16<Bf16> {};
template <>
struct Oct<Fp16> : Oct16<Fp16> {};
template <>
struct Oct<F32Elt> {
  typedef float type;
  static __device__ __forceinline__ void get(const type* p, long i, float (&v)[8]) {
    const float4 lo = *reinterpret_cast<const float4*>(p + i), hi = *reinterpret_cast<const float4*>(p + i + 4);
    v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w; v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
  }
  static __device__ __forceinline__ void put(type* p, long i, const float (&v)[8]) {
    *reinterpret_cast<float4*>(p + i) = make_float4(v[0], v[1], v[2], v[3]);
    *reinterpret_cast<float4*>(p + i + 4) = make_float4(v[4], v[5], v[6], v[7]);
  }
};

struct StepScalars {
  float a, r_new, r_store;
};

// Per-head scalar update: gate, inclusive in-block gate product (linear or log accumulator).
__device__ __forceinline__ StepScalars step_scalars(const JagStepArgs& p, long row) {
  StepScalars s;
  const float A = load_scalar(p.a_t, row, p.a_dtype);
  s.a = p.log_a ? __expf(A) : A;
  const float prev = p.r_in != nullptr ? load_scalar(p.r_in, row, p.r_dtype) : (p.log_r ? 0.0f : 1.0f);
  if (p.log_r) {
    const float lr = prev + __logf(fmaxf(s.a, p.tiny));
    s.r_new = __expf(lr);
    s.r_store = lr;
  } else {
    s.r_new = s.a * prev;
    s.r_store = s.r_new;
  }
  if (p.boundary) s.r_store = p.log_r ? 0.0f : 1.0f;
  return s;
}

template <class T, class S>
__global__ __launch_bounds__(256) void jagged_step_kernel(const JagStepArgs p, long octs, int octs_per_head) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= octs) return;
  const long row = idx / octs_per_head;
  const long e = idx * 8;
  typedef typename Oct<T>::type elt_t;
  typedef typename Oct<S>::type st_t;

  const StepScalars s = step_scalars(p, row);
  float h[8], x[8], cp[8], y[8], c[8], v[8];
  Oct<S>::get(static_cast<const st_t*>(p.h_in), e, h);
  Oct<S>::get(static_cast<const st_t*>(p.c_prev_in), e, cp);
  Oct<T>::get(static_cast<const elt_t*>(p.x_t), e, x);
  const bool epilogue = p.c_t != nullptr;  // its two loads go out with the others, ahead of any arithmetic
  if (epilogue) {
    Oct<T>::get(static_cast<const elt_t*>(p.c_t), e, c);
    Oct<T>::get(static_cast<const elt_t*>(p.v_t), e, v);
  }
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    h[q] = s.a * h[q] + x[q];
    y[q] = h[q] + s.r_new * cp[q];
  }
  if (epilogue) {
#pragma unroll
    for (int q = 0; q < 8; ++q) y[q] = y[q] * c[q] + v[q];
  }
  Oct<T>::put(static_cast<elt_t*>(p.y_t), e, y);
  if (p.boundary) {
    Oct<S>::put(static_cast<st_t*>(p.c_prev_out), e, h);
#pragma unroll
    for (int q = 0; q < 8; ++q) h[q] = 0.0f;
  }
  Oct<S>::put(static_cast<st_t*>(p.h_out), e, h);
  if (idx % octs_per_head == 0) store_scalar(p.r_out, row, p.r_dtype, s.r_store);
}

// Any head size: one thread per head walks its channels (never races, whatever aliases).
template <class T, class S>
__global__ __launch_bounds__(256) void jagged_step_any_kernel(const JagStepArgs p, long rows, int D) {
  const long row = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= rows) return;
  typedef typename Scalar<T>::type elt_t;
  typedef typename Scalar<S>::type st_t;
  const StepScalars s = step_scalars(p, row);
  for (int d = 0; d < D; ++d) {
    const long e = row * D + d;
    const float h = s.a * Scalar<S>::get(static_cast<const st_t*>(p.h_in), e) + Scalar<T>::get(static_cast<const elt_t*>(p.x_t), e);
    float yv = h + s.r_new * Scalar<S>::get(static_cast<const st_t*>(p.c_prev_in), e);
    if (p.c_t != nullptr)
      yv = yv * Scalar<T>::get(static_cast<const elt_t*>(p.c_t), e) + Scalar<T>::get(static_cast<const elt_t*>(p.v_t), e);
    Scalar<T>::put(static_cast<elt_t*>(p.y_t), e, yv);
    if (p.boundary) Scalar<S>::put(static_cast<st_t*>(p.c_prev_out), e, h);
    Scalar<S>::put(static_cast<st_t*>(p.h_out), e, p.boundary ? 0.0f : h);
  }
  store_scalar(p.r_out, row, p.r_dtype, s.r_store);
}

template <class T, class S>
hipError_t launch_step(const JagStepArgs& p, hipStream_t s) {
  const long rows = (long)p.B * p.H;
  // the 8-channel form needs whole octets per head, and heads whose threads share a wavefront
  // (64 % octets == 0) so that an aliased scalar is read by all of them before it is written
  const int oph = p.D / 8;
  if (p.aligned && p.D % 8 == 0 && 64 % oph == 0) {
    const long octs = rows * oph;
    hipLaunchKernelGGL((jagged_step_kernel<T, S>), dim3((unsigned)((octs + 255) / 256)), dim3(256), 0, s, p, octs, oph);
  } else {
    hipLaunchKernelGGL((jagged_step_any_kernel<T, S>), dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, s, p, rows, p.D);
  }
  return hipGetLastError();
}

template <class T>
hipError_t step_by_state(const JagStepArgs& p, hipStream_t s) {
  if (p.state_dtype == p.x_dtype) return launch_step<T, T>(p, s);
  return launch_step<T, F32Elt>(p, s);  // validated by the caller: otherwise fp32 state
}

template <class E, class C>
void launch_prefill_tiled(const JagPrefillArgs& p, hipStream_t s) {
  const Grid g = make_grid((long)p.B * p.H, p.L);
  const auto* a = static_cast<const typename C::elem*>(p.a);
  const auto* x = static_cast<const uint16_t*>(p.x);
  const auto* c = static_cast<const uint16_t*>(p.c);
  const auto* v = static_cast<const uint16_t*>(p.v);
  auto* y = static_cast<uint16_t*>(p.y);
  const bool st = stream_inputs(g);
  auto word_aligned = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 3u) == 0; };
  const bool on_words = word_aligned(p.x) && word_aligned(p.c) && word_aligned(p.v) && word_aligned(p.y);
  const int align = (p.L % 8 == 0 && p.aligned) ? 16 : !on_words ? 2 : (p.L % 2 == 0) ? 4 : 1;
#define SPEAR_JAG_LAUNCH(EPI, ST, AL)                                                                         \
  hipLaunchKernelGGL((jagged_prefill_kernel<E, C, EPI, ST, AL>), dim3(g.blocks), dim3(64 * kWaves), 0, s, a, x, \
                     c, v, p.carry_init, y, p.h_tail, p.r_tail, p.c_prev_tail, p.state_dtype, p.r_dtype, p.L,   \
                     g.spans_per_row, g.total_spans)
#define SPEAR_JAG_BY_SPAN(EPI, AL) \
  do {                             \
    if (st) SPEAR_JAG_LAUNCH(EPI, true, AL); \
    else SPEAR_JAG_LAUNCH(EPI, false, AL);   \
  } while (0)
#define SPEAR_JAG_BY_ALIGN(EPI)                       \
  do {                                                \
    if (align == 16) SPEAR_JAG_BY_SPAN(EPI, 16);      \
    else if (align == 4) SPEAR_JAG_BY_SPAN(EPI, 4);   \
    else if (align == 1) SPEAR_JAG_BY_SPAN(EPI, 1);   \
    else SPEAR_JAG_BY_SPAN(EPI, 2);                   \
  } while (0)
  if (p.c != nullptr) SPEAR_JAG_BY_ALIGN(true);
  else SPEAR_JAG_BY_ALIGN(false);
#undef SPEAR_JAG_BY_ALIGN
#undef SPEAR_JAG_BY_SPAN
#undef SPEAR_JAG_LAUNCH
}

template <class T>
void launch_prefill_any(const JagPrefillArgs& p, hipStream_t s) {
  typedef typename Scalar<T>::type elt_t;
  const long rows = (long)p.B * p.H;
  const int nblk = (p.L + p.block_len - 1) / p.block_len;
  const long threads = rows * p.D * nblk;
  hipLaunchKernelGGL((jagged_prefill_any_kernel<T>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, p.a,
                     p.a_dtype, p.log_a ? 1 : 0, static_cast<const elt_t*>(p.x), static_cast<const elt_t*>(p.c),
                     static_cast<const elt_t*>(p.v), p.carry_init, static_cast<elt_t*>(p.y), p.h_tail, p.r_tail,
                     p.c_prev_tail, p.state_dtype, p.r_dtype, rows, p.D, p.L, p.block_len, nblk);
}


// Longest block the tile kernel takes: its image holds two blocks of 16 channel rows in fp32 and their gates per wavefront, 34.25 KiB
// at 256 steps, and four wavefronts' images have to fit the 160 KiB of a compute unit.
constexpr int kMaxTileBlock = 256;

// How blocks of `block_len` <= L steps make a tile: about 64 steps, as at most four lane groups of whole blocks. Tiles of 128 steps measured
// the same or slower: 177 -> 184 us in fp32 at B=1024 H=32 L=128, 78 us either way in bf16 at B=16 H=16 D=64 L=2048 in blocks of 64.
struct TileShape {
  int per_lane, lanes, width, spans;  // blocks per lane group, lane groups, steps of a tile, tiles per row
};
TileShape tile_shape(int block_len, int L) {
  constexpr int steps = 64;
  TileShape t;
  t.per_lane = block_len < steps / 4 ? steps / 4 / block_len : 1;
  const int chunk = t.per_lane * block_len;
  t.lanes = chunk > steps ? 1 : steps / chunk > 4 ? 4 : steps / chunk;
  t.width = t.lanes * chunk;
  t.spans = (L + t.width - 1) / t.width;
  return t;
}

template <class T, int kG, int kN>
hipError_t launch_tile_as(const TileArgs& t, bool shared, hipStream_t s) {
  const size_t lds = (size_t)kTileWaves * t.wave_floats * sizeof(float);
  const dim3 grid((unsigned)((t.tiles + kTileWaves - 1) / kTileWaves)), block(64 * kTileWaves);
  auto go = [&](auto kernel) {
    if (lds > 64 * 1024) {  // above the default limit of dynamic LDS
      const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (err != hipSuccess) return err;
    }
    hipLaunchKernelGGL(kernel, grid, block, lds, s, t);
    return hipGetLastError();
  };
  if (!shared) return go(jagged_prefill_tile_kernel<T, kG, kN, false, 0>);
  if (t.block_len == 16) return go(jagged_prefill_tile_kernel<T, kG, kN, true, 16>);
  return go(jagged_prefill_tile_kernel<T, kG, kN, true, 0>);
}

template <class T>
hipError_t launch_prefill_tile(const JagPrefillArgs& p, hipStream_t s) {
  constexpr int kBytes = sizeof(typename Scalar<T>::type);
  TileArgs t{};
  t.coeff = p.a; t.x = p.x; t.c = p.c; t.v = p.v; t.carry_init = p.carry_init;
  t.y = p.y; t.h_tail = p.h_tail; t.r_tail = p.r_tail; t.c_prev_tail = p.c_prev_tail;
  t.rd_total = (long)p.B * p.H * p.D;
  t.tensor_bytes = t.rd_total * p.L * kBytes;
  t.D = p.D; t.L = p.L; t.whole = p.block_len;
  const int block_len = t.block_len = p.block_len < p.L ? p.block_len : p.L;
  t.nblk = (p.L + block_len - 1) / block_len;
  t.a_dtype = p.a_dtype; t.log_a = p.log_a ? 1 : 0; t.state_dtype = p.state_dtype; t.r_dtype = p.r_dtype;
  // The widest granule whose grid every row of every tensor (and, with block lengths on that grid, every tile of a row)
  // starts on.
  auto all_on = [&](int bytes) {
    auto on = [&](const void* q) { return (reinterpret_cast<uintptr_t>(q) % bytes) == 0; };
    return on(p.x) && on(p.c) && on(p.v) && on(p.y);
  };
  const bool wide = all_on(16) && ((long)p.L * kBytes) % 16 == 0 && (block_len * kBytes) % 16 == 0;
  const int granule = wide ? 16 : all_on(4) ? 4 : 2;
  const int per_granule = granule / kBytes;
  const TileShape shape = tile_shape(block_len, p.L);
  t.per_lane = shape.per_lane;
  t.lanes = shape.lanes;
  t.spans = shape.spans;
  const int W = shape.width, pad = (block_len + 3) & ~3;
  t.tiles = (t.rd_total + kTileRows - 1) / kTileRows * t.spans;
  const int chunks = (pad + W + 3) / 4;
  t.stride = 4 * (chunks | 1);  // an odd number of 16-byte chunks: 16 rows' reads of one column spread over the banks
  t.wave_floats = kTileRows * t.stride + 4 * chunks;
  // a 16-bit row that starts on a word's second half covers one word more
  const int extra = kBytes == 2 && granule == 4 ? 1 : 0;
  t.main_gpr = (W + per_granule - 1) / per_granule + extra;
  t.halo_gpr = (block_len + per_granule - 1) / per_granule + extra;
  t.main_magic = ((1u << 20) + t.main_gpr - 1) / t.main_gpr;
  t.halo_magic = ((1u << 20) + t.halo_gpr - 1) / t.halo_gpr;
  const bool shared = p.D % kTileRows == 0;  // a tile's channel rows then share one gate row
  if (granule == 16) return launch_tile_as<T, 16, kBytes>(t, shared, s);
  if constexpr (kBytes == 4) {
    return launch_tile_as<T, 4, 16>(t, shared, s);
  } else {
    if (granule == 4) return launch_tile_as<T, 4, 9>(t, shared, s);
    return launch_tile_as<T, 2, 16>(t, shared, s);
  }
}

// Which kernel a prompt takes. A tile has room for about 64 steps of a row and its lanes walk whole blocks, so rows and blocks of few steps
// leave much of it idle; one thread per block is wasteful where its neighbours' words lie far apart (long blocks) and the tensors
// are larger than the L2 caches. Tile kernel / one thread per block, us, D=16 (16 channel rows share a gate row) and D=5 (they don't):
//   fp32, 128 MiB per tensor: L=96 in blocks of 16 85 / 1446, 197 / 1518; of 8 86 / 481, 166 / 504; of 4 86 / 238, 142 / 248; of 2
//     130 / 169, 209 / 171; L=9 in blocks of 9 or more 507 / 650, 877 / 672 (bf16 2.3 and 2.7 times as long in tiles)
//   fp32, 2 MiB: L=96 in blocks of 16 5.1 / 14.8, 11.1 / 15.4; of 8 5.5 / 8.5, 10.2 / 8.7; of 4 5.7 / 6.1, 9.2 / 6.1
//   bf16, 8 MiB: L=96 in blocks of 8 10.5 / 31.8, 17.7 / 38.6; of 4 18.1 / 18.0, 24.3 / 18.6
// Over 9960 forms (L 5 to 1000, blocks of 1 to 200, D 1, 5, 16, 1 to 128 MiB, fp32 and bf16) the rule takes the slower kernel by more than
// 3 % in 12, by 20 % at most (D=5, rows of 19), and 0.72 of the time of one thread per block in the geometric mean; the faster
// one of the two each time would be 0.66, tiles throughout 0.93.
bool tiles_pay_off(const JagPrefillArgs& p, int block_len, long row_bytes) {
  const TileShape t = tile_shape(block_len, p.L);
  const bool shared = p.D % kTileRows == 0, big = (long)p.B * p.H * p.D * row_bytes >= (8L << 20);
  const double used = (double)p.L / ((double)t.spans * t.width);  // of the tiles' columns
  if (block_len >= 16) return big || (shared && used >= 0.45);
  if (block_len >= 8) return big && used >= 0.6;
  return block_len >= 4 && big && shared && used >= 0.8;
}

// The tile kernel's limits: 32-bit offsets inside the 16 rows of a tile, and a grid of 31 bits
template <class T>
hipError_t launch_prefill_general(const JagPrefillArgs& p, hipStream_t s) {
  const long row_bytes = (long)p.L * (long)sizeof(typename Scalar<T>::type);
  const int block_len = p.block_len < p.L ? p.block_len : p.L;  // of a lane's work: rows shorter than a block end before it does
  const long tiles_at_most = ((long)p.B * p.H * p.D / kTileRows + 1) * ((p.L + block_len - 1) / block_len);
  if (block_len <= kMaxTileBlock && row_bytes * (kTileRows + 1) < 0x70000000L && tiles_at_most < (1L << 31) &&
      tiles_pay_off(p, block_len, row_bytes))
    return launch_prefill_tile<T>(p, s);
  launch_prefill_any<T>(p, s);
  return hipGetLastError();
}
}  // namespace

bool jagged_prefill_is_tiled(const JagPrefillArgs& p) {
  const bool own16 = p.a_dtype == p.x_dtype;        // a_t or log(a_t) in the tensors' 16-bit type
  const bool log32 = p.log_a && p.a_dtype == kF32;  // fp32 log-space gate
  return p.x_dtype != kF32 && p.D == kChan && p.block_len == kTile && (own16 || log32);
}

hipError_t jagged_prefill(const JagPrefillArgs& p, hipStream_t s) {
  if (jagged_prefill_is_tiled(p)) {
    if (p.x_dtype == kBf16) {
      if (!p.log_a) launch_prefill_tiled<Bf16, LinCoeff<Bf16>>(p, s);
      else if (p.a_dtype == kF32) launch_prefill_tiled<Bf16, LogCoeff>(p, s);
      else launch_prefill_tiled<Bf16, LogCoeff16<Bf16>>(p, s);
    } else {
      if (!p.log_a) launch_prefill_tiled<Fp16, LinCoeff<Fp16>>(p, s);
      else if (p.a_dtype == kF32) launch_prefill_tiled<Fp16, LogCoeff>(p, s);
      else launch_prefill_tiled<Fp16, LogCoeff16<Fp16>>(p, s);
    }
    return hipGetLastError();
  }
  if (p.x_dtype == kBf16) return launch_prefill_general<Bf16>(p, s);
  if (p.x_dtype == kF16) return launch_prefill_general<Fp16>(p, s);
  return launch_prefill_general<F32Elt>(p, s);
}

hipError_t jagged_step(const JagStepArgs& p, hipStream_t s) {
  if (p.x_dtype == kBf16) return step_by_state<Bf16>(p, s);
  if (p.x_dtype == kF16) return step_by_state<Fp16>(p, s);
  return launch_step<F32Elt, F32Elt>(p, s);
}

}  // namespace spear_btp
