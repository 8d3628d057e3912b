// What the layer's large matrix kernels share: 16-byte loads from memory to LDS, waits and barriers that the compiler leaves where they
// are, and the matrix instruction.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

// The asm blocks below write m0, which the compiler keeps for itself and sets anew before each of its own uses.
#pragma clang diagnostic ignored "-Winline-asm"

namespace spear_btp {

namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void lds_void_t;

// An offset past the end of every buffer: loads give zero there and stores are dropped. Offsets of up to 2^30 may be added to it.
constexpr uint32_t kNowhere = 0x80000000u;

__device__ __forceinline__ f32x4_t mfma(i32x4_t a, i32x4_t b, f32x4_t acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), acc, 0, 0, 0);
}

// acc[i][j] += w[j] x[i] over 32 columns of K.
template <int kRowTiles, int kColTiles>
__device__ __forceinline__ void multiply(f32x4_t (&acc)[kRowTiles][kColTiles], const i32x4_t (&w)[kColTiles], const i32x4_t (&x)[kRowTiles]) {
#pragma unroll
  for (int j = 0; j < kColTiles; ++j)
#pragma unroll
    for (int i = 0; i < kRowTiles; ++i) acc[i][j] = mfma(w[j], x[i], acc[i][j]);
}

// The same where `first` says that a quarter of K starts here: the sums so far go to `sum` and acc starts again, beside the matrix instructions.
template <int kRowTiles, int kColTiles>
__device__ __forceinline__ void multiply_quarters(f32x4_t (&acc)[kRowTiles][kColTiles], f32x4_t (&sum)[kRowTiles][kColTiles],
                                                  const i32x4_t (&w)[kColTiles], const i32x4_t (&x)[kRowTiles], bool first) {
  if (first) {
#pragma unroll
    for (int j = 0; j < kColTiles; ++j)
#pragma unroll
      for (int i = 0; i < kRowTiles; ++i) {
        sum[i][j] += acc[i][j];
        acc[i][j] = mfma(w[j], x[i], f32x4_t{0.0f, 0.0f, 0.0f, 0.0f});
      }
  } else {
    multiply(acc, w, x);
  }
}

// A buffer of `bytes` bytes (none if negative), which the hardware checks every access against.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, max(bytes, 0), 0x00020000);
}

// The same descriptor as four words, for asm.
__device__ __forceinline__ i32x4_t words_of(const void* p, int bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  return i32x4_t{(int)(uint32_t)a, (int)(uint32_t)(a >> 32 & 0xffff), max(bytes, 0), 0x00020000};
}

// Four requests inside an asm block, counted by wait_vm: 16 bytes per lane from the buffer of `desc` at the lane's offset (o0 .. o3, checked against the
// buffer's size) + `further` (sgpr, not checked) to 16 lane past LDS addresses 1 KiB apart from `lds` on (sgpr). A write of m0 has to be one
// instruction ahead of its use.
#define SPEAR_REQUEST4(lds, o0, o1, o2, o3, desc, further)                                            \
  "s_mov_b32 m0, " lds "\n s_nop 0\n buffer_load_dwordx4 " o0 ", " desc ", " further " offen lds\n"    \
  "s_add_u32 m0, " lds ", 0x400\n s_nop 0\n buffer_load_dwordx4 " o1 ", " desc ", " further " offen lds\n" \
  "s_add_u32 m0, " lds ", 0x800\n s_nop 0\n buffer_load_dwordx4 " o2 ", " desc ", " further " offen lds\n" \
  "s_add_u32 m0, " lds ", 0xc00\n s_nop 0\n buffer_load_dwordx4 " o3 ", " desc ", " further " offen lds\n"

#define SPEAR_REQUEST2(lds, o0, o1, desc, further)                                                   \
  "s_mov_b32 m0, " lds "\n s_nop 0\n buffer_load_dwordx4 " o0 ", " desc ", " further " offen lds\n"     \
  "s_add_u32 m0, " lds ", 0x400\n s_nop 0\n buffer_load_dwordx4 " o1 ", " desc ", " further " offen lds\n"

__device__ __forceinline__ uint32_t lds_address(char* p) { return (uint32_t)(uintptr_t)(lds_void_t*)p; }

// Until no more than kOutstanding of this wavefront's loads and stores are under way.
template <int kOutstanding>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kOutstanding) : "memory");
}

// A barrier that no instruction is moved over. It orders LDS only with the waits that the caller has made: fragment reads end with
// theirs, loads to LDS with wait_vm.
__device__ __forceinline__ void phase_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

constexpr int kRowsStep = 64;  // columns of K asked for at a time

// One operand's rows of a tile, asked for 64 columns of K at a time: the lane's offsets of four requests (rows 8 apart; a row's pieces are
// exchanged by ((row >> 1) & 7), so that the reads of a fragment touch every bank once), and what is left of K.
struct Rows {
  i32x4_t of;             // descriptor, ends with the tile's last row
  uint32_t at[4], piece;
  int further, left;      // bytes of a row asked for, and left
};

__device__ __forceinline__ void aim(Rows& r, const uint16_t* first, int rows, int ld, int K) {
  r.of = words_of(first, ((rows - 1) * ld + K) * 2);
  r.further = 0;
  r.left = 2 * K;
}

// Ahead of the request that meets the end of K: nowhere from there on. The empty asm keeps this, and what else is done a few times per tile,
// out of the steps between (the compiler would work it out every time and select).
__device__ __forceinline__ void end_rows(Rows& r) {
  if (r.left < 2 * kRowsStep) {
    asm volatile("");
#pragma unroll
    for (int i = 0; i < 4; ++i) r.at[i] = (int)(i & 1 ? r.piece ^ 64 : r.piece) < r.left ? r.at[i] : kNowhere;
  }
}

__device__ __forceinline__ void advance(Rows& r) {
  r.further += 2 * kRowsStep;
  r.left -= 2 * kRowsStep;
}

// The next 64 columns into LDS from address `to` on.
__device__ __forceinline__ void request(Rows& r, uint32_t to) {
  asm volatile(SPEAR_REQUEST4("%4", "%0", "%1", "%2", "%3", "%5", "%6")
               :: "v"(r.at[0]), "v"(r.at[1]), "v"(r.at[2]), "v"(r.at[3]), "s"(to), "s"(r.of), "s"(r.further) : "memory", "m0", "scc");
  advance(r);
}

}  // namespace

}  // namespace spear_btp
