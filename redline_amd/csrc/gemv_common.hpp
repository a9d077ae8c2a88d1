// Device pieces shared by the weight-only GEMV kernels (gemv_w4.hip and
// gemv_stream.hip): launch arguments, code conversion, the output epilogue.
#pragma once

#include <hip/hip_runtime.h>

#include "device.hpp"
#include "redline_amd/rlk.h"
#include "status.hpp"

namespace rlk {
namespace {

struct W4Args {
  const uint16_t* x;  // activations of this launch, [m, k]
  const uint8_t* w;
  const uint16_t* scales;
  const uint16_t* offsets;
  const uint16_t* bias;
  void* y;            // [m, y_ld]
  int m;              // activation rows (1 .. 16 MT)
  int n, k, group_size, groups, nchunks;
  int cpp;            // K chunks per x pass (a multiple of K-split ways x ring depth);
                      // K-slice kernel: 16-row tiles per workgroup
  int npass;
  int xstride;        // halves per staged x row
  int slab_off;       // bytes from the end of x to the first chunk-pair slab;
                      // K-slice kernel: bytes from the LDS base to the partial sums
  int y_ld;
  int gq_shift;       // pair kernel: log2(group_size / 128)
  int gpp;            // pair kernel: quantisation groups per x pass
};

constexpr int kModeF16 = 0, kModeF32 = 1, kModeSwiglu = 2;
constexpr int kSlabRow = 144;                // bytes per slab row: 128 code bytes + 16 pad
constexpr int kSlabBytes = 16 * kSlabRow;    // one wave's chunk-pair slab

// Codes of one lane for one chunk: 32 K (16 bytes) for 128-K chunks, 8 K
// (4 bytes) for 32-K chunks.  Weights are read exactly once: non-temporal.
template <int KC>
__device__ __forceinline__ u32x4 load_codes(const uint8_t* p) {
  if constexpr (KC == 128) {
    return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
  } else {
    u32x4 v = {__builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(p)), 0u, 0u, 0u};
    return v;
  }
}

// A value the compiler must keep in a VGPR without knowing it (the empty asm
// emits no instruction).  With the code magic opaque, (x & mask) | magic is
// selected as one v_and_or_b32 (mask in an SGPR); with both operands known
// constants the compiler splits it into AND + OR, because gfx9 VOP3
// encodings take no literal.  Writing the op itself as inline asm would hide
// it from the compiler's hazard recognizer, which must pad a VALU write of an
// MFMA source operand.
__device__ __forceinline__ uint32_t opaque(uint32_t v) {
  asm volatile("" : "+v"(v));
  return v;
}

__device__ __forceinline__ uint32_t and_or(uint32_t x, uint32_t mask, uint32_t magic) {
  return (x & mask) | magic;
}

// The 8 codes of a word (nibble e = code of K offset e) as fp16 values
// 64 + q, in the order (q0, q4, q1, q5, q2, q6, q3, q7): a nibble placed in
// mantissa bits 4..7 of 64.0 (0x5400) reads 64 + q exactly.  The bias of 64
// is removed through the offset term (o - 64 s), computed once per group in
// fp32; it keeps the MFMA sums within a small factor of the unbiased ones.
__device__ __forceinline__ f16x8 codes_f16(uint32_t word, uint32_t magic) {
  constexpr uint32_t kMask = 0x00F000F0u;
  const u32x4 r = {and_or(word << 4, kMask, magic), and_or(word, kMask, magic),
                   and_or(word >> 4, kMask, magic), and_or(word >> 8, kMask, magic)};
  return __builtin_bit_cast(f16x8, r);
}
constexpr float kCodeBias = 64.0f;

// The same values in K order (q0, q1, ..., q7), for activations as they lie in
// memory: one shift, then per pair a byte permute (the even nibble's byte from
// the shifted word, the odd one's from the word) and the masked OR: 9 VALU per
// word where codes_f16 takes 7 and 4 more for each 8 activations (x_perm).
__device__ __forceinline__ f16x8 codes_f16_natural(uint32_t word, uint32_t magic) {
  constexpr uint32_t kMask = 0x00F000F0u;
  const uint32_t even = word << 4;  // byte i: nibble 2 i in its upper half
  const u32x4 r = {and_or(__builtin_amdgcn_perm(word, even, 0x0C040C00u), kMask, magic),
                   and_or(__builtin_amdgcn_perm(word, even, 0x0C050C01u), kMask, magic),
                   and_or(__builtin_amdgcn_perm(word, even, 0x0C060C02u), kMask, magic),
                   and_or(__builtin_amdgcn_perm(word, even, 0x0C070C03u), kMask, magic)};
  return __builtin_bit_cast(f16x8, r);
}

// The K-slice kernel's form: 5 VALU per 8 codes instead of 7.  Nibbles in
// mantissa bits 0..3 of 1024.0 read 1024 + q, in bits 4..7 of 64.0 read
// 64 + q, so the word needs one shift: (q0, q4) and (q2, q6) take magic
// m1024, (q1, q5) and (q3, q7) m64 -- the same element order as codes_f16.
// The biases leave through sum(x * kBias2) per chunk.  The larger bias costs
// fp32 sum bits (the kernel's relative error grows from ~1.5e-6 to ~2e-5 at
// k = 4096; the fp32-output bound is 1e-4).
__device__ __forceinline__ f16x8 codes_f16_2m(uint32_t word, uint32_t m1024, uint32_t m64) {
  const uint32_t w8 = word >> 8;
  const u32x4 r = {and_or(word, 0x000F000Fu, m1024), and_or(word, 0x00F000F0u, m64),
                   and_or(w8, 0x000F000Fu, m1024), and_or(w8, 0x00F000F0u, m64)};
  return __builtin_bit_cast(f16x8, r);
}
// The bias of each element of codes_f16_2m's output.
constexpr f16x8 kBias2 = {1024, 1024, 64, 64, 1024, 1024, 64, 64};

// 8 consecutive activations permuted to the codes' order.
__device__ __forceinline__ f16x8 x_perm(u32x4 v) {
  const f16x8 h = __builtin_bit_cast(f16x8, v);
  return __builtin_shufflevector(h, h, 0, 4, 1, 5, 2, 6, 3, 7);
}

// v / d for 0 <= v < 2^21 through a float reciprocal: (v + 1/2) / d lies at
// least 1/(2d) away from an integer and the float error is below 2^-22 * v/d.
__device__ __forceinline__ int quot(int v, float inv_d) {
  return static_cast<int>((static_cast<float>(v) + 0.5f) * inv_d);
}

__device__ __forceinline__ float swap_adjacent_lanes(float v) {
  // quad_perm (1, 0, 3, 2): each lane reads its odd/even neighbour
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0xB1, 0xF,
                                                            0xF, false));
}

// Output of one 16x16 tile: lane (qd, r16) holds rows m = m0 + 4 qd + e of
// weight row `row`; b is that row's bias.
template <int MODE>
__device__ __forceinline__ void store_tile(const W4Args& a, f32x4 v, float b, int m0, int row, int r16) {
  if constexpr (MODE == kModeSwiglu) {
    // (gate, up) = rows (2i, 2i + 1) sit in lanes (r16, r16 + 1)
    f32x4 up;
#pragma unroll
    for (int e = 0; e < 4; ++e) up[e] = swap_adjacent_lanes(v[e]);
    if ((r16 & 1) != 0 || row >= a.n) return;
    uint16_t* y = static_cast<uint16_t*>(a.y) + row / 2;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (m0 + e >= a.m) break;
      const float g = round_f16(v[e]);
      const float u = round_f16(up[e]);
      y[static_cast<size_t>(m0 + e) * a.y_ld] =
          __builtin_bit_cast(uint16_t, static_cast<_Float16>(silu_f16(g) * u));
    }
  } else {
    if (row >= a.n) return;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (m0 + e >= a.m) break;
      const size_t at = static_cast<size_t>(m0 + e) * a.y_ld + row;
      if constexpr (MODE == kModeF32) {
        static_cast<float*>(a.y)[at] = v[e] + b;
      } else {
        static_cast<uint16_t*>(a.y)[at] = __builtin_bit_cast(uint16_t, static_cast<_Float16>(v[e] + b));
      }
    }
  }
}

// The bias of weight row `row` (0 without one, or past n).
__device__ __forceinline__ float row_bias(const W4Args& a, int row) {
  return a.bias != nullptr && row < a.n ? static_cast<float>(__builtin_bit_cast(_Float16, a.bias[row])) : 0.f;
}
template <int MODE>
__device__ __forceinline__ void store_tile(const W4Args& a, f32x4 v, int m0, int row, int r16) {
  if constexpr (MODE == kModeSwiglu) {
    store_tile<MODE>(a, v, 0.f, m0, row, r16);
  } else {
    if (row >= a.n) return;
    store_tile<MODE>(a, v, row_bias(a, row), m0, row, r16);
  }
}

constexpr int kMaxWaves = 8;  // of a workgroup: two waves per SIMD, up to 256 VGPRs each
// Word 3 of a buffer resource for raw byte-addressed loads (32-bit data
// format, no swizzle), and the cache-policy operand of the buffer-load
// builtins that marks a load non-temporal.
constexpr int kBufferFlags = 0x00020000;
constexpr int kNtLoad = 2;
// Largest weight addressed through 32-bit buffer offsets.
constexpr uint64_t kMaxBufferBytes = 0x7FFFFFFFu;
// LDS a workgroup may take: the device allows 160 KiB per workgroup.
constexpr size_t kLdsBudget = 160 * 1024;
constexpr int kNoFit = 1;  // a launcher's kernel does not take this shape

}  // namespace
}  // namespace rlk
