// fp32 / bf16 MFMA tile helpers for gfx950 (v_mfma_f32_32x32x2f32,
// v_mfma_f32_16x16x4f32, v_mfma_f32_32x32x16_bf16) shared by the chunk kernels.
//
// Operand feeding.  A 32x32x2 MFMA step takes one A and one B value per lane:
// A(row l%32, c), B(c, col l%32) with c = 2 s + l/32.  mma8 instead feeds,
// over four steps s = 0..3, contraction index c0 + s with c0 = 8 g + 4 (l/32):
// the same 8 indices of group g, permuted.  A lane then needs four consecutive
// contraction values of one row or column: one vector LDS read when the
// contraction axis is contiguous (ld_c), four conflict-free scalar reads when
// the row axis is (ld_x).  The accumulator of a 32x32 tile holds, in lane l
// register r, row 8 (r/4) + 4 (l/32) + r%4 and column l%32 (acc_row); the
// bf16 32x32x16 MFMA uses the same accumulator layout with lane l holding row
// (or column) l%32 and contraction indices 8 (l/32) .. +7 of each 16-step.
#pragma once
#include <hip/hip_runtime.h>

#include "gdn_common.h"

namespace gpa {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));


__device__ __forceinline__ void mma8(f32x16& c, f32x4 a, f32x4 b) {
  c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b.x, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b.y, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, b.z, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, b.w, c, 0, 0, 0);
}

// 16x16x4 with the same permutation: lane quarter q = l/16 feeds c0 + s, c0 = 16 g + 4 q.
__device__ __forceinline__ void mma16(f32x4& c, f32x4 a, f32x4 b) {
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, c, 0, 0, 0);
}

// Element (x, c0 + s), s = 0..3, of a matrix stored with c contiguous ...
__device__ __forceinline__ f32x4 ld_c(const float* m, int ld, int x, int c0) {
  return *reinterpret_cast<const f32x4*>(m + x * ld + c0);
}
// ... or with x contiguous.
__device__ __forceinline__ f32x4 ld_x(const float* m, int ld, int x, int c0) {
  return f32x4{m[c0 * ld + x], m[(c0 + 1) * ld + x], m[(c0 + 2) * ld + x], m[(c0 + 3) * ld + x]};
}

// The operands of mma16 with the contraction indices in order: its MFMAs are chains of
// fused multiply-adds over the quarters, so with index c0 + 4 s + l/16 in element s the
// sum runs over c0, c0 + 1, ...  Where the terms of neighbouring indices cancel (the
// delta rule's over positions, when keys are nearly parallel), any other order adds up
// large partial sums first.
__device__ __forceinline__ f32x4 ld_c_inorder(const float* m, int ld, int x, int c0, int q) {
  const float* p = m + x * ld + c0 + q;
  return f32x4{p[0], p[4], p[8], p[12]};
}
__device__ __forceinline__ f32x4 ld_x_inorder(const float* m, int ld, int x, int c0, int q) {
  const float* p = m + (c0 + q) * ld + x;
  return f32x4{p[0], p[4 * ld], p[8 * ld], p[12 * ld]};
}

__device__ __forceinline__ int acc_row(int r, int half) { return 8 * (r >> 2) + 4 * half + (r & 3); }

// x of lanes 32..63 trades places with y of lanes 0..31 ...
__device__ __forceinline__ void swap_halves(uint32_t& x, uint32_t& y) {
  const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
  x = r[0];
  y = r[1];
}
// ... and x of lanes 16..31, 48..63 with y of lanes 0..15, 32..47.
__device__ __forceinline__ void swap_quarters(uint32_t& x, uint32_t& y) {
  const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
  x = r[0];
  y = r[1];
}
// Elements 4 (l/16) + e of an accumulator column to elements 4 e + l/16 (the B operand of
// the next product, its indices in order), by an exchange of quarters and elements.
__device__ __forceinline__ f32x4 acc_inorder(f32x4 x) {
  uint32_t u[4];
  __builtin_memcpy(u, &x, 16);
  swap_halves(u[0], u[2]);
  swap_halves(u[1], u[3]);
  swap_quarters(u[0], u[1]);
  swap_quarters(u[2], u[3]);
  __builtin_memcpy(&x, u, 16);
  return x;
}
// The value of another lane of the row of 16: l ^ 8, l ^ 7, l ^ 3, l ^ 2, l ^ 1.
constexpr int DPP_XOR8 = 0x128, DPP_XOR7 = 0x141, DPP_XOR3 = 0x1b, DPP_XOR2 = 0x4e, DPP_XOR1 = 0xb1;
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  return __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), CTRL, 0xf, 0xf, false));
}

__device__ __forceinline__ uint32_t dpp_xor4(uint32_t x) {
  return __builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp(x, DPP_XOR7, 0xf, 0xf, false), DPP_XOR3, 0xf, 0xf, false);
}
__device__ __forceinline__ float dpp_xor4(float x) { return __uint_as_float(dpp_xor4(__float_as_uint(x))); }
// Eight consecutive lanes hold the rows of an 8 x 8 bf16 matrix; returns its
// columns the same way.  Bits 2 and 1 of the row trade places with the dword
// index, bit 0 with the half of a dword.
__device__ __forceinline__ uint4 transpose8_lanes(uint4 v, int lane) {
  uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const bool up = lane & 4;
    const uint32_t got = dpp_xor4(up ? d[i] : d[i + 2]);
    d[i] = up ? got : d[i];
    d[i + 2] = up ? d[i + 2] : got;
  }
#pragma unroll
  for (int i = 0; i < 4; i += 2) {
    const bool up = lane & 2;
    const uint32_t got = __builtin_amdgcn_mov_dpp(up ? d[i] : d[i + 1], DPP_XOR2, 0xf, 0xf, false);
    d[i] = up ? got : d[i];
    d[i + 1] = up ? d[i + 1] : got;
  }
  const uint32_t sel = lane & 1 ? 0x07060302u : 0x01000504u;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    d[i] = __builtin_amdgcn_perm(d[i], __builtin_amdgcn_mov_dpp(d[i], DPP_XOR1, 0xf, 0xf, false), sel);
  return make_uint4(d[0], d[1], d[2], d[3]);
}

// Sums of each of a lane's 16 accumulator-row values over the 32 lanes of its
// half-wave, by recursive halving (lanes l ^ 16, 8, 4, 2, 1) without LDS.
// Every lane returns the sum for register index sum_index(lane).
__device__ __forceinline__ float tile_row_sum(float (&v)[16], int lane) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    uint32_t x = __float_as_uint(v[j]), y = __float_as_uint(v[j + 8]);
    swap_quarters(x, y);
    v[j] = __uint_as_float(x) + __uint_as_float(y);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const bool up = lane & 8;
    const float send = up ? v[j] : v[j + 4], keep = up ? v[j + 4] : v[j];
    v[j] = keep + dpp<DPP_XOR8>(send);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const bool up = lane & 4;
    const float send = up ? v[j] : v[j + 2], keep = up ? v[j + 2] : v[j];
    v[j] = keep + dpp_xor4(send);
  }
  const bool up = lane & 2;
  const float send = up ? v[0] : v[1], keep = up ? v[1] : v[0];
  v[0] = keep + dpp<DPP_XOR2>(send);
  return v[0] + dpp<DPP_XOR1>(v[0]);
}
__device__ __forceinline__ int sum_index(int lane) {
  return 8 * ((lane >> 4) & 1) + 4 * ((lane >> 3) & 1) + 2 * ((lane >> 2) & 1) + ((lane >> 1) & 1);
}

// Four consecutive activation-type elements as floats (8 bytes for bf16).
__device__ __forceinline__ f32x4 ld_c(const bf16_t* m, int ld, int x, int c0) {
  const uint2 w = *reinterpret_cast<const uint2*>(m + x * ld + c0);
  return f32x4{__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u), __uint_as_float(w.y << 16),
               __uint_as_float(w.y & 0xffff0000u)};
}

template <typename E>
__device__ __forceinline__ E op_raw(const gpa_operand& o, int b, int h, int t, int d) {
  return reinterpret_cast<const E*>(o.ptr)[op_base(o, b, h) + (int64_t)t * o.st + d];
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Eight consecutive floats rounded to bf16 (round to nearest even).
__device__ __forceinline__ bf16x8 pack8(const float* x) {
  const f32x4 a = *reinterpret_cast<const f32x4*>(x), c = *reinterpret_cast<const f32x4*>(x + 4);
  bf16x8 r;
  r[0] = (__bf16)a.x; r[1] = (__bf16)a.y; r[2] = (__bf16)a.z; r[3] = (__bf16)a.w;
  r[4] = (__bf16)c.x; r[5] = (__bf16)c.y; r[6] = (__bf16)c.z; r[7] = (__bf16)c.w;
  return r;
}

// Split bf16 operands of v_mfma_f32_32x32x16_bf16 (lane l: row or column
// l%32, contraction 8 (l/32) .. +7).  An fp32 value x is carried as hi + lo,
// hi = bf16(x), lo = bf16(x - hi); a product keeps hi*hi + hi*lo + lo*hi,
// about 16 significant bits.  Values exact in bf16 go in unsplit.
struct SplitBf8 {
  bf16x8 hi, lo;
};
// Eight floats as bf16 hi and lo vectors (element e of x is element e of each).
__device__ __forceinline__ void split8(const float (&x)[8], bf16x8& hi, bf16x8& lo) {
  uint32_t h[4], o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) bf2_split(x[2 * i], x[2 * i + 1], h[i], o[i]);
  __builtin_memcpy(&hi, h, 16);
  __builtin_memcpy(&lo, o, 16);
}
// Rows 16 gp .. 16 gp + 15 of an accumulator tile, eight consecutive rows per
// lane (those + 8 in the upper lanes), split into bf16 hi and lo.
__device__ __forceinline__ SplitBf8 split_rows(const f32x16& acc, int gp) {
  float v[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t x = __float_as_uint(acc[8 * gp + i]), y = __float_as_uint(acc[8 * gp + 4 + i]);
    swap_halves(x, y);
    v[i] = __uint_as_float(x);
    v[4 + i] = __uint_as_float(y);
  }
  SplitBf8 s;
  split8(v, s.hi, s.lo);
  return s;
}
__device__ __forceinline__ SplitBf8 split_bf8(const float (&x)[8]) {
  SplitBf8 s;
  split8(x, s.hi, s.lo);
  return s;
}
// Elements (c0 + e, x), e = 0..7, of an fp32 matrix stored with x contiguous.
__device__ __forceinline__ SplitBf8 col_split_bf8(const float* m, int ld, int x, int c0) {
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = m[(c0 + e) * ld + x];
  return split_bf8(v);
}
// Elements (x, c0 + e) of an fp32 matrix stored with c contiguous (16-byte aligned rows).
__device__ __forceinline__ SplitBf8 row_split_bf8(const float* m, int ld, int x, int c0) {
  const f32x4 a = *reinterpret_cast<const f32x4*>(m + x * ld + c0), b = *reinterpret_cast<const f32x4*>(m + x * ld + c0 + 4);
  const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  return split_bf8(v);
}
// Elements (x, c0 + e) of a bf16 matrix stored with c contiguous (8-byte aligned rows).
__device__ __forceinline__ bf16x8 row_bf8(const bf16_t* m, int ld, int x, int c0) {
  const uint2 a = *reinterpret_cast<const uint2*>(m + x * ld + c0), b = *reinterpret_cast<const uint2*>(m + x * ld + c0 + 4);
  const uint4 w = make_uint4(a.x, a.y, b.x, b.y);
  bf16x8 r;
  __builtin_memcpy(&r, &w, 16);
  return r;
}
__device__ __forceinline__ void mma_bf16(f32x16& c, bf16x8 a, bf16x8 b) {
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ void mma_split(f32x16& c, const SplitBf8& a, const SplitBf8& b) {
  mma_bf16(c, a.hi, b.hi);
  mma_bf16(c, a.hi, b.lo);
  mma_bf16(c, a.lo, b.hi);
}
__device__ __forceinline__ void mma_exact_split(f32x16& c, bf16x8 a, const SplitBf8& b) {
  mma_bf16(c, a, b.hi);
  mma_bf16(c, a, b.lo);
}
__device__ __forceinline__ void mma_split_exact(f32x16& c, const SplitBf8& a, bf16x8 b) {
  mma_bf16(c, a.hi, b);
  mma_bf16(c, a.lo, b);
}

}  // namespace gpa
