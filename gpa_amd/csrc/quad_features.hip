// Quadratic Q/K feature map (reference src/gpa/features.py:17-25), forward and
// backward, one workgroup per (32-row tile, head):
//   u = unit(x) rounded to E;  a = u L, b = u R (E products, float32 accumulation,
//   rounded to E);  z = u + (c a) b with c = 2 sigmoid(gain_raw) sqrt(D);
//   out = unit(z) ||x||_eps rounded to E.
// The two products run on the MFMA (v_mfma_f32_32x32x16_bf16 for bf16,
// v_mfma_f32_32x32x2f32 for float32) with u staged in LDS and the weights read
// as 16-byte rows of a transposed, zero-padded copy (the caller prepares it:
// the weights are parameters, a few hundred KB).  Wave w owns the column
// blocks w, w + 4 of both products, so a and b of an element meet in one
// lane's accumulators; row sums go through the half-wave and LDS.
//
// The backward recomputes the forward, forms dz through the two
// normalisations, da = (dz b) c and db = dz (c a) rounded to E, and
// du = dz + da L^T + db R^T as one MFMA product over the concatenated
// [da | db] rows; dx follows through unit(x) and ||x||.  It also writes u and
// [da | db] head-major for the weight gradients u^T [da | db] (bf16:
// gpa_quad_weight_grads, two launches; float32: a batched product the caller
// runs) and one partial sum of dc per workgroup.
#include <hip/hip_runtime.h>

#include <initializer_list>

#include "mfma_tiles.h"

namespace gpa {
namespace {

constexpr int QT = 256;   // threads per workgroup (4 waves)
constexpr int QR = 32;    // rows per workgroup
// (column blocks per wave, QB: 1 up to 128 columns, else 2)

__host__ __device__ inline int qpad(int d) { return (d + 31) / 32 * 32; }
__device__ __forceinline__ int qmin(int a, int b) { return a < b ? a : b; }

// LDS: rows of u, and for the backward of x, dout (then dx) and [da | db], each
// row padded by 16 bytes; per-row scalars.
template <typename E>
struct QLayout {
  int DP, NB, ULD, DLD;
  E* u;         // [32][ULD] unit(x) rows, then the output rows (out, dx)
  E* x;         // [32][ULD] raw rows, zeros past dim and past the last row (null: q_raw_in_lds)
  E* g;         // [32][ULD] dout rows, the same, in dab's place until dab is formed
  E* dab;       // [32][DLD] d(a) | d(b) rows
  float* nrm;   // [32] ||x||_eps = sqrt(sum x^2 + 1e-12)
  float* xn;    // [32] sqrt(sum x^2)
  float* part;  // [2][8][32] per-block row partial sums
  float* ra;    // [32] row values of the phase at hand
  float* rb;
  float* dn;    // [32] d ||x||_eps
  float* wsum;  // [4] per-wave partial of dc
};

// Whether the backward keeps the raw rows in LDS: not in float32 above 128 columns, where
// they would leave one workgroup per compute unit instead of two up to 192 columns
// (8192 rows x 16 heads, forward and backward: 130 columns 1161 us with them, 869 without,
// 192 columns 1443 and 1206; 256 columns, one either way, 1826 and 1846); they are read
// again there.
template <typename E>
__host__ __device__ constexpr bool q_raw_in_lds(int dim) { return sizeof(E) == 2 || dim <= 128; }

template <typename E>
__host__ __device__ inline size_t q_lds_bytes(int dim, bool backward) {
  const int DP = qpad(dim), ULD = DP + 16 / (int)sizeof(E), DLD = 2 * DP + 16 / (int)sizeof(E);
  const int rows = backward && q_raw_in_lds<E>(dim) ? 2 : 1;
  const size_t b = (size_t)QR * ULD * sizeof(E) * rows + (backward ? (size_t)QR * DLD * sizeof(E) : 0);
  return b + (5 * QR + 16 * QR + 4) * sizeof(float);
}

template <typename E>
__device__ QLayout<E> q_layout(char* smem, int dim, bool backward) {
  QLayout<E> L;
  L.DP = qpad(dim);
  L.NB = L.DP / 32;
  L.ULD = L.DP + 16 / (int)sizeof(E);
  L.DLD = 2 * L.DP + 16 / (int)sizeof(E);
  E* e = reinterpret_cast<E*>(smem);
  L.u = e;
  e += QR * L.ULD;
  L.x = nullptr;
  if (backward) {
    if (q_raw_in_lds<E>(dim)) {
      L.x = e;
      e += QR * L.ULD;
    }
    L.g = L.dab = e;
    e += QR * L.DLD;
  }
  float* f = reinterpret_cast<float*>(e);
  L.nrm = f;
  L.xn = f + QR;
  L.ra = f + 2 * QR;
  L.rb = f + 3 * QR;
  L.dn = f + 4 * QR;
  L.part = f + 5 * QR;
  L.wsum = f + 21 * QR;
  return L;
}

// One 16-byte piece of a row of E.
template <typename E>
struct QPiece {
  static constexpr int N = 16 / sizeof(E);
  E v[N];
};
template <typename E>
__device__ __forceinline__ QPiece<E> q_get(const E* src) {
  const uint4 w = *reinterpret_cast<const uint4*>(src);
  QPiece<E> x;
  __builtin_memcpy(&x, &w, 16);
  return x;
}
__device__ __forceinline__ bool q_aligned(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }
template <typename E>
__device__ __forceinline__ void q_put(E* dst, const QPiece<E>& x) {
  uint4 w;
  __builtin_memcpy(&w, &x, 16);
  *reinterpret_cast<uint4*>(dst) = w;
}
// Rows r0 .. r0+31 of `src`, `stride` apart, to LDS (zero past dim and past the last
// row), element-wise: a wave per row, a lane per element of 64, so that rows off
// 16-byte boundaries are read in whole lines too (8192 x 16 rows of 250 bf16, forward and
// backward: 651 us; 785 with each thread on its own pieces' elements).
template <typename E>
__device__ __forceinline__ void q_stage(const gpa_quad_problem& p, const E* src, int64_t stride, int r0,
                                        const QLayout<E>& L, E* dst) {
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, D = p.dim;
  for (int c = l; c < L.DP; c += 64) {
    E v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = src[qmin(r0 + 8 * w + i, p.rows - 1) * stride + qmin(c, D - 1)];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      dst[(8 * w + i) * L.ULD + c] = r0 + 8 * w + i < p.rows && c < D ? v[i] : from_f32<E>(0.f);
  }
}

// Rows r0 .. r0+31 of head h: u into LDS (zero past dim and past the last row)
// and, with ROWS, the raw rows (RAW) and dout's, u also to `uo`; ||x|| and ||x||_eps per
// row.  Thread t holds the 16-byte pieces t%8, t%8 + 8, ... of row t/8, loaded as such
// (VEC; every load is issued before the first use) or from the rows in LDS.
template <typename E, bool VEC, bool ROWS, bool RAW>
__device__ void q_rows(const gpa_quad_problem& p, const E* dout, E* uo, int h, int r0, QLayout<E>& L) {
  constexpr int N = QPiece<E>::N, PM = 256 / (8 * N);
  const int tid = threadIdx.x, row = tid / 8, part = tid % 8, D = p.dim;
  const bool live = r0 + row < p.rows;
  const int grow = live ? r0 + row : p.rows - 1;
  const E* xh = reinterpret_cast<const E*>(p.x) + (int64_t)h * D;
  const E* gh = ROWS ? dout + (int64_t)h * D : nullptr;
  const int64_t gs = (int64_t)p.heads * D;
  constexpr bool PUT = VEC && ROWS;  // dout's pieces are not in LDS yet
  E* raw = RAW ? L.x : L.u;
  QPiece<E> xv[PM], gv[PUT ? PM : 1];
  if constexpr (VEC) {
#pragma unroll
    for (int i = 0; i < PM; ++i) {
      const int d = (part + 8 * i) * N;
      xv[i] = q_get(xh + grow * p.row_stride + (d < D ? d : 0));
    }
    if constexpr (ROWS)
#pragma unroll
      for (int i = 0; i < PM; ++i) {
        const int d = (part + 8 * i) * N;
        gv[i] = q_get(gh + grow * gs + (d < D ? d : 0));
      }
  } else {
    q_stage(p, xh, p.row_stride, r0, L, raw);
    if constexpr (ROWS) q_stage(p, gh, gs, r0, L, L.g);
    lds_barrier();
#pragma unroll
    for (int i = 0; i < PM; ++i) {
      const int d = (part + 8 * i) * N;
      xv[i] = q_get(raw + row * L.ULD + (d < L.DP ? d : 0));
    }
  }
  if constexpr (VEC) {
#pragma unroll
    for (int i = 0; i < PM; ++i) {
      const int d = (part + 8 * i) * N;
#pragma unroll
      for (int e = 0; e < N; ++e) {
        const bool ok = live && d + e < D;
        if (!ok) xv[i].v[e] = from_f32<E>(0.f);
        if constexpr (PUT)
          if (!ok) gv[i].v[e] = from_f32<E>(0.f);
      }
      if (d < L.DP) q_put(raw + row * L.ULD + d, xv[i]);
    }
    lds_barrier();
  }
  // The sum of squares: elements t%8, t%8 + 8, ... in order, then the eight lanes.
  float ss = 0.f;
#pragma unroll 4
  for (int i = 0; i < L.DP / 8; ++i) {
    const float x = to_f32(raw[row * L.ULD + part + 8 * i]);
    ss += x * x;
  }
  ss += __shfl_xor(ss, 1, 64);
  ss += __shfl_xor(ss, 2, 64);
  ss += __shfl_xor(ss, 4, 64);
  const float n = sqrtf(ss), den = fmaxf(n, 1e-6f);
#pragma unroll
  for (int i = 0; i < PM; ++i) {
    const int d = (part + 8 * i) * N;
    if (d >= L.DP) continue;
    if constexpr (PUT) q_put(L.g + row * L.ULD + d, gv[i]);
#pragma unroll
    for (int e = 0; e < N; ++e) xv[i].v[e] = from_f32<E>(to_f32(xv[i].v[e]) / den);
    q_put(L.u + row * L.ULD + d, xv[i]);
    if constexpr (ROWS)
      if (live) {  // (u has whole pieces whatever the width)
        E* dst = uo + ((int64_t)h * p.rows + r0 + row) * L.DP + d;
        if (VEC || q_aligned(uo)) q_put(dst, xv[i]);
        else
          for (int e = 0; e < N; ++e) dst[e] = xv[i].v[e];
      }
  }
  if (part == 0) {
    L.nrm[row] = sqrtf(ss + 1e-12f);
    L.xn[row] = n;
  }
}

// Rows in LDS (from `src`, `ld` apart) to `width` elements of the live rows of
// dst, `stride` apart: in 16-byte pieces (vec) or, as in q_stage, element-wise.
template <typename E>
__device__ __forceinline__ void q_rows_out(const gpa_quad_problem& p, int r0, E* dst, int64_t stride, int width,
                                           const E* src, int ld, bool vec) {
  if (vec) {
    constexpr int N = QPiece<E>::N;
    const int row = threadIdx.x / 8;
    if (r0 + row < p.rows)
      for (int d = (threadIdx.x % 8) * N; d < width; d += 8 * N) q_put(dst + row * stride + d, q_get(src + row * ld + d));
  } else {
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    for (int row = 8 * w; row < 8 * w + 8 && r0 + row < p.rows; ++row)
      for (int c = l; c < width; c += 64) dst[row * stride + c] = src[row * ld + c];
  }
}

// A per-row array at a lane's accumulator rows.
__device__ __forceinline__ void q_at_rows(const float* a, float (&x)[16]) {
  const int hi = (threadIdx.x & 63) >> 5;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(a + 8 * g + 4 * hi);
#pragma unroll
    for (int i = 0; i < 4; ++i) x[4 * g + i] = v[i];
  }
}

// acc_a, acc_b = u W_p for the 32 columns of block cb (p = 0: left, 1: right).
template <typename E>
__device__ __forceinline__ void q_products(const gpa_quad_problem& p, int h, int cb, const QLayout<E>& L,
                                           f32x16& acc_a, f32x16& acc_b) {
  const int l = threadIdx.x & 63, lr = l & 31, hi = l >> 5;
  const E* wt = reinterpret_cast<const E*>(p.wt);
  const E* wl = wt + ((int64_t)(h * 2 + 0) * L.DP + cb * 32 + lr) * L.DP;
  const E* wr = wt + ((int64_t)(h * 2 + 1) * L.DP + cb * 32 + lr) * L.DP;
  for (int i = 0; i < 16; ++i) acc_a[i] = acc_b[i] = 0.f;
  if constexpr (sizeof(E) == 2) {
    const bf16_t* u = reinterpret_cast<const bf16_t*>(L.u);
    for (int ks = 0; ks < L.DP / 16; ++ks) {
      const int k0 = 16 * ks + 8 * hi;
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(u + lr * L.ULD + k0);
      const bf16x8 bl = *reinterpret_cast<const bf16x8*>(wl + k0);
      const bf16x8 br = *reinterpret_cast<const bf16x8*>(wr + k0);
      mma_bf16(acc_a, a, bl);
      mma_bf16(acc_b, a, br);
    }
  } else {
    const float* u = reinterpret_cast<const float*>(L.u);
    for (int ks = 0; ks < L.DP / 8; ++ks) {
      const int c0 = 8 * ks + 4 * hi;
      const f32x4 a = ld_c(u, L.ULD, lr, c0);
      const f32x4 bl = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(wl) + c0);
      const f32x4 br = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(wr) + c0);
      mma8(acc_a, a, bl);
      mma8(acc_b, a, br);
    }
  }
}

// Row sums of a lane's 16 accumulator-layout values over the block's 32
// columns, into part[cb][row].
__device__ __forceinline__ void q_row_part(float (&v)[16], float* part, int cb) {
  const int l = threadIdx.x & 63;
  const float s = tile_row_sum(v, l);
  if ((l & 1) == 0) part[cb * QR + acc_row(sum_index(l), l >> 5)] = s;
}
__device__ __forceinline__ float q_row_total(const float* part, int nb, int r) {
  float s = 0.f;
  for (int cb = 0; cb < nb; ++cb) s += part[cb * QR + r];
  return s;
}

// z (and a, b) at a wave's elements of column block cb; its squares' row sums.
template <typename E>
__device__ __forceinline__ void q_z(const gpa_quad_problem& p, int h, int cb, const QLayout<E>& L, float c,
                                    float (&z)[16], float (&av)[16], float (&bv)[16]) {
  const int l = threadIdx.x & 63;
  f32x16 acc_a, acc_b;
  q_products<E>(p, h, cb, L, acc_a, acc_b);
  float zz[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    av[r] = round_as<E>(acc_a[r]);
    bv[r] = round_as<E>(acc_b[r]);
    z[r] = to_f32(L.u[acc_row(r, l >> 5) * L.ULD + cb * 32 + (l & 31)]) + (c * av[r]) * bv[r];
    zz[r] = z[r] * z[r];
  }
  q_row_part(zz, L.part, cb);
}

// Rows move between HBM and LDS in 16-byte pieces, a row per 8 lanes, and the
// per-row values of an elementwise phase (roots, cubes) are formed once per row
// by 32 threads; the divisions stay per element, since a reciprocal per row rounds
// otherwise (3 and 15 us less, but other bits).  Bound: HBM (the backward moves 6 rows of dim
// per row) and those divisions; element-wise 2-byte accesses and a root per element before.
// bf16, 8192 rows x 16 heads x 128: forward 67 -> 52 us, backward 210 -> 104 us.
// VEC: dim a whole number of 16-byte pieces, every row on a 16-byte boundary.
template <typename E, bool VEC, int QB>
__global__ __launch_bounds__(QT) void quad_fwd(gpa_quad_problem p) {
  extern __shared__ __align__(16) char smem[];
  const int h = blockIdx.y, r0 = blockIdx.x * QR, w = threadIdx.x >> 6, l = threadIdx.x & 63;
  QLayout<E> L = q_layout<E>(smem, p.dim, false);
  q_rows<E, VEC, false, false>(p, nullptr, nullptr, h, r0, L);
  lds_barrier();
  const float c = p.gain[h];
  float z[QB][16];
#pragma unroll
  for (int bi = 0; bi < QB; ++bi) {
    if (w + 4 * bi >= L.NB) break;
    float a[16], b[16];
    q_z<E>(p, h, w + 4 * bi, L, c, z[bi], a, b);
  }
  lds_barrier();
  if (threadIdx.x < QR)
    L.ra[threadIdx.x] = fmaxf(sqrtf(q_row_total(L.part, L.NB, threadIdx.x)), 1e-6f);
  lds_barrier();
  float zn[16], nrm[16];
  q_at_rows(L.ra, zn);
  q_at_rows(L.nrm, nrm);
#pragma unroll
  for (int bi = 0; bi < QB; ++bi) {
    const int cb = w + 4 * bi;
    if (cb >= L.NB) break;
#pragma unroll
    for (int r = 0; r < 16; ++r) L.u[acc_row(r, l >> 5) * L.ULD + cb * 32 + (l & 31)] = from_f32<E>(z[bi][r] / zn[r] * nrm[r]);
  }
  lds_barrier();
  q_rows_out(p, r0, reinterpret_cast<E*>(p.out) + ((int64_t)r0 * p.heads + h) * p.dim, (int64_t)p.heads * p.dim, p.dim,
             L.u, L.ULD, VEC);
}

template <typename E, bool VEC, int QB>
__global__ __launch_bounds__(QT) void quad_bwd(gpa_quad_problem p, gpa_quad_grads g) {
  extern __shared__ __align__(16) char smem[];
  const int h = blockIdx.y, r0 = blockIdx.x * QR, w = threadIdx.x >> 6, l = threadIdx.x & 63, t = threadIdx.x;
  const int D = p.dim;
  QLayout<E> L = q_layout<E>(smem, D, true);
  constexpr bool RAW = q_raw_in_lds<E>(128 * QB);
  q_rows<E, VEC, true, RAW>(p, reinterpret_cast<const E*>(g.dout), reinterpret_cast<E*>(g.u), h, r0, L);
  lds_barrier();
  const float c = p.gain[h];
  float z[QB][16], av[QB][16], bv[QB][16], gv[QB][16];
  auto at = [&](int r, int cb) { return acc_row(r, l >> 5) * L.ULD + cb * 32 + (l & 31); };
#pragma unroll
  for (int bi = 0; bi < QB; ++bi) {
    const int cb = w + 4 * bi;
    if (cb >= L.NB) break;
    q_z<E>(p, h, cb, L, c, z[bi], av[bi], bv[bi]);
#pragma unroll
    for (int r = 0; r < 16; ++r) gv[bi][r] = to_f32(L.g[at(r, cb)]);
  }
  lds_barrier();
  if (t < QR) L.ra[t] = fmaxf(sqrtf(q_row_total(L.part, L.NB, t)), 1e-6f);
  lds_barrier();
  // out = unit(z) nrm: d nrm = sum g unit(z), d unit(z) = g nrm; the
  // normalisation backward needs sum d unit(z) . z per row.
  {
    float zn[16], nrm[16];
    q_at_rows(L.ra, zn);
    q_at_rows(L.nrm, nrm);
#pragma unroll
    for (int bi = 0; bi < QB; ++bi) {
      const int cb = w + 4 * bi;
      if (cb >= L.NB) break;
      float s1[16], s2[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s1[r] = gv[bi][r] * (z[bi][r] / zn[r]);
        gv[bi][r] *= nrm[r];
        s2[r] = gv[bi][r] * z[bi][r];
      }
      q_row_part(s1, L.part, cb);
      q_row_part(s2, L.part + 8 * QR, cb);
    }
  }
  lds_barrier();
  if (t < QR) {  // dz = g nrm / ra - z rb
    const float zt = L.ra[t];
    L.dn[t] = q_row_total(L.part, L.NB, t);
    L.rb[t] = q_row_total(L.part + 8 * QR, L.NB, t) / (zt * zt * zt);
  }
  lds_barrier();
  // dz, then da = (dz b) c, db = dz (c a) in E; du starts as dz rounded to E.
  float dc = 0.f;
  {
    float ra[16], rb[16];
    q_at_rows(L.ra, ra);
    q_at_rows(L.rb, rb);
#pragma unroll
    for (int bi = 0; bi < QB; ++bi) {
      const int cb = w + 4 * bi;
      if (cb >= L.NB) break;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float du = gv[bi][r] / ra[r];
        const float dz = ra[r] > 1e-6f ? du - z[bi][r] * rb[r] : du;
        const float t1 = dz * bv[bi][r];
        dc += t1 * av[bi][r];
        E* d = L.dab + acc_row(r, l >> 5) * L.DLD + cb * 32 + (l & 31);
        d[0] = from_f32<E>(t1 * c);
        d[L.DP] = from_f32<E>(dz * (c * av[bi][r]));
        z[bi][r] = round_as<E>(dz);
      }
    }
  }
  dc = sum64(dc);
  if (l == 0) L.wsum[w] = dc;
  lds_barrier();
  if (t == 0) g.dgain[(int64_t)blockIdx.x * p.heads + h] = L.wsum[0] + L.wsum[1] + L.wsum[2] + L.wsum[3];
  q_rows_out(p, r0, reinterpret_cast<E*>(g.dab) + ((int64_t)h * p.rows + r0) * 2 * L.DP, 2 * L.DP, 2 * L.DP, L.dab, L.DLD,
             VEC || q_aligned(g.dab));
  // du = dz + da L^T + db R^T: contraction over the 2 DP columns of [da | db];
  // the B operand of output column k is row k of w = [L | R] (contiguous).
  const E* wk = reinterpret_cast<const E*>(p.w);
#pragma unroll
  for (int bi = 0; bi < QB; ++bi) {
    const int cb = w + 4 * bi;
    if (cb >= L.NB) break;
    f32x16 acc_l, acc_r;
    for (int i = 0; i < 16; ++i) acc_l[i] = acc_r[i] = 0.f;
    const int lr = l & 31, hi = l >> 5;
    const E* wrow = wk + ((int64_t)h * L.DP + cb * 32 + lr) * 2 * L.DP;
    if constexpr (sizeof(E) == 2) {
      const bf16_t* d = reinterpret_cast<const bf16_t*>(L.dab);
      for (int ks = 0; ks < L.DP / 16; ++ks) {
        const int k0 = 16 * ks + 8 * hi;
        mma_bf16(acc_l, *reinterpret_cast<const bf16x8*>(d + lr * L.DLD + k0),
                 *reinterpret_cast<const bf16x8*>(wrow + k0));
        mma_bf16(acc_r, *reinterpret_cast<const bf16x8*>(d + lr * L.DLD + L.DP + k0),
                 *reinterpret_cast<const bf16x8*>(wrow + L.DP + k0));
      }
    } else {
      const float* d = reinterpret_cast<const float*>(L.dab);
      const float* wf = reinterpret_cast<const float*>(wrow);
      for (int ks = 0; ks < L.DP / 8; ++ks) {
        const int c0 = 8 * ks + 4 * hi;
        mma8(acc_l, ld_c(d, L.DLD, lr, c0), *reinterpret_cast<const f32x4*>(wf + c0));
        mma8(acc_r, ld_c(d, L.DLD, lr, L.DP + c0), *reinterpret_cast<const f32x4*>(wf + L.DP + c0));
      }
    }
    float s3[16];
    if constexpr (!RAW) {
      const int col = cb * 32 + lr;
      const E* xh = reinterpret_cast<const E*>(p.x) + (int64_t)h * D + qmin(col, D - 1);
#pragma unroll
      for (int r = 0; r < 16; ++r) av[bi][r] = to_f32(xh[qmin(r0 + acc_row(r, l >> 5), p.rows - 1) * p.row_stride]);
#pragma unroll
      for (int r = 0; r < 16; ++r) av[bi][r] = r0 + acc_row(r, l >> 5) < p.rows && col < D ? av[bi][r] : 0.f;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      if constexpr (RAW) av[bi][r] = to_f32(L.x[at(r, cb)]);
      z[bi][r] = round_as<E>(z[bi][r] + round_as<E>(acc_l[r]) + round_as<E>(acc_r[r]));
      s3[r] = z[bi][r] * av[bi][r];
    }
    q_row_part(s3, L.part, cb);
  }
  lds_barrier();
  if (t < QR) {  // dx = du / ra - x rb, through unit(x), + dn x / nrm, through ||x||_eps
    const float n = fmaxf(L.xn[t], 1e-6f);
    L.ra[t] = n;
    L.rb[t] = q_row_total(L.part, L.NB, t) / (n * n * n);
  }
  lds_barrier();
  float ra[16], rb[16], dn[16], nrm[16];
  q_at_rows(L.ra, ra);
  q_at_rows(L.rb, rb);
  q_at_rows(L.dn, dn);
  q_at_rows(L.nrm, nrm);
#pragma unroll
  for (int bi = 0; bi < QB; ++bi) {
    const int cb = w + 4 * bi;
    if (cb >= L.NB) break;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float x = av[bi][r], du = z[bi][r] / ra[r];
      const float d = ra[r] > 1e-6f ? du - x * rb[r] : du;
      L.u[at(r, cb)] = from_f32<E>(d + dn[r] * x / nrm[r]);
    }
  }
  lds_barrier();
  q_rows_out(p, r0, reinterpret_cast<E*>(g.dx) + ((int64_t)r0 * p.heads + h) * D, (int64_t)p.heads * D, D, L.u, L.ULD, VEC);
}

// The two weight layouts from the float32 parameters [H][D][D], a 32 x 32 tile per
// workgroup: wt transposed through LDS, w (may be null) as read; zeros past D.
// One launch in place of a stack, a cast, a pad and two strided copies (19 us each
// at 16 heads x 128).
template <typename E>
__global__ __launch_bounds__(QT) void quad_pack(const float* left, const float* right, E* wt, E* w, int D) {
  __shared__ float tile[32][33];
  const int DP = qpad(D), NB = DP / 32, h = blockIdx.y, p = blockIdx.x & 1, tb = blockIdx.x >> 1;
  const int k0 = tb / NB * 32, n0 = tb % NB * 32, c = threadIdx.x % 32, r0 = threadIdx.x / 32;
  const float* src = (p ? right : left) + (int64_t)h * D * D;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int k = k0 + r0 + 8 * i, n = n0 + c;
    const bool ok = k < D && n < D;
    const float x = src[ok ? (int64_t)k * D + n : 0];
    tile[r0 + 8 * i][c] = ok ? x : 0.f;
    if (w) w[((int64_t)h * DP + k) * 2 * DP + p * DP + n] = from_f32<E>(ok ? x : 0.f);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i)
    wt[(((int64_t)h * 2 + p) * DP + n0 + r0 + 8 * i) * DP + k0 + c] = from_f32<E>(tile[c][r0 + 8 * i]);
}

int check_quad(const gpa_quad_problem* pp) {
  if (!pp) return fail(GPA_HIP_EINVAL, "quad features: null problem");
  const gpa_quad_problem& p = *pp;
  if (p.rows < 1 || p.heads < 1 || p.dim < 1 || p.dim > GPA_QUAD_MAX_DIM)
    return fail(GPA_HIP_EINVAL, "quad features: rows, heads positive, dim 1..GPA_QUAD_MAX_DIM");
  if (p.dtype != GPA_DTYPE_F32 && p.dtype != GPA_DTYPE_BF16) return fail(GPA_HIP_EUNSUPPORTED, "quad features: dtype");
  if (!p.x || !p.wt || !p.w || !p.gain || p.row_stride < (int64_t)p.heads * p.dim)
    return fail(GPA_HIP_EINVAL, "quad features: x, wt, w, gain required; row_stride >= heads*dim");
  if ((int64_t)(p.rows + QR - 1) / QR > 0x7fffffff || p.heads > 65535)
    return fail(GPA_HIP_EINVAL, "quad features: too many rows or heads");
  return 0;
}

template <typename K, typename... A>
int q_launch(K kernel, const gpa_quad_problem& p, size_t lds, hipStream_t stream, A... args) {
  if (lds > 65536 && hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return fail(GPA_HIP_EHIP, "hipFuncSetAttribute(max dynamic LDS) failed");
  const dim3 grid((unsigned)((p.rows + QR - 1) / QR), (unsigned)p.heads);
  hipLaunchKernelGGL(kernel, grid, dim3(QT), lds, stream, p, args...);
  return 0;
}

// Every row of these buffers starts on a 16-byte boundary and is a whole
// number of 16-byte pieces.
template <typename E>
bool q_vec(const gpa_quad_problem& p, std::initializer_list<const void*> buffers) {
  const int n = 16 / (int)sizeof(E);
  bool ok = p.dim % n == 0 && p.row_stride % n == 0;
  for (const void* b : buffers) ok = ok && reinterpret_cast<uintptr_t>(b) % 16 == 0;
  return ok;
}

template <typename E>
int q_forward(const gpa_quad_problem& p, hipStream_t stream) {
  const size_t lds = q_lds_bytes<E>(p.dim, false);
  const bool vec = q_vec<E>(p, {p.x, p.out});
  if (p.dim <= 128) return q_launch(vec ? quad_fwd<E, true, 1> : quad_fwd<E, false, 1>, p, lds, stream);
  return q_launch(vec ? quad_fwd<E, true, 2> : quad_fwd<E, false, 2>, p, lds, stream);
}
template <typename E>
int q_backward(const gpa_quad_problem& p, const gpa_quad_grads& g, hipStream_t stream) {
  const size_t lds = q_lds_bytes<E>(p.dim, true);
  const bool vec = q_vec<E>(p, {p.x, g.dout, g.dx, g.u, g.dab});
  if (p.dim <= 128) return q_launch(vec ? quad_bwd<E, true, 1> : quad_bwd<E, false, 1>, p, lds, stream, g);
  return q_launch(vec ? quad_bwd<E, true, 2> : quad_bwd<E, false, 2>, p, lds, stream, g);
}

}  // namespace
}  // namespace gpa

extern "C" int gpa_quad_features_forward(const gpa_quad_problem* problem, hipStream_t stream) {
  using namespace gpa;
  if (int rc = check_quad(problem)) return rc;
  if (!problem->out) return fail(GPA_HIP_EINVAL, "quad features: out required");
  if (int rc = problem->dtype == GPA_DTYPE_BF16 ? q_forward<bf16_t>(*problem, stream) : q_forward<float>(*problem, stream))
    return rc;
  return check_launch("gpa_quad_features_forward");
}

extern "C" int gpa_quad_features_backward(const gpa_quad_problem* problem, const gpa_quad_grads* grads,
                                          hipStream_t stream) {
  using namespace gpa;
  if (int rc = check_quad(problem)) return rc;
  if (!grads || !grads->dout || !grads->dx || !grads->u || !grads->dab || !grads->dgain)
    return fail(GPA_HIP_EINVAL, "quad features backward: dout, dx, u, dab and dgain required");
  if (int rc = problem->dtype == GPA_DTYPE_BF16 ? q_backward<bf16_t>(*problem, *grads, stream)
                                                : q_backward<float>(*problem, *grads, stream))
    return rc;
  return check_launch("gpa_quad_features_backward");
}

extern "C" int gpa_quad_pack_weights(const float* left, const float* right, int32_t heads, int32_t dim, int32_t dtype,
                                     void* wt, void* w, hipStream_t stream) {
  using namespace gpa;
  if (!left || !right || !wt || heads < 1 || heads > 65535 || dim < 1 || dim > GPA_QUAD_MAX_DIM)
    return fail(GPA_HIP_EINVAL, "quad pack: left, right, wt required; heads 1..65535, dim 1..GPA_QUAD_MAX_DIM");
  if (dtype != GPA_DTYPE_F32 && dtype != GPA_DTYPE_BF16) return fail(GPA_HIP_EUNSUPPORTED, "quad pack: dtype");
  const int nb = qpad(dim) / 32;
  const dim3 grid(2 * nb * nb, heads);
  if (dtype == GPA_DTYPE_BF16)
    hipLaunchKernelGGL((quad_pack<bf16_t>), grid, dim3(QT), 0, stream, left, right, static_cast<bf16_t*>(wt),
                       static_cast<bf16_t*>(w), dim);
  else
    hipLaunchKernelGGL((quad_pack<float>), grid, dim3(QT), 0, stream, left, right, static_cast<float*>(wt),
                       static_cast<float*>(w), dim);
  return check_launch("gpa_quad_pack_weights");
}

namespace gpa {
namespace {
// dW_p[h] = sum over the rows of u^T da (p = 0), u^T db (p = 1).
struct QuadProducts {
  TnProduct p[2];
  QuadProducts(const gpa_quad_problem& q, const void* u, const void* dab, float* dleft, float* dright) {
    const int dp = qpad(q.dim);
    const int64_t hs = (int64_t)q.rows * dp;
    const bf16_t* b = static_cast<const bf16_t*>(dab);
    p[0] = {u, dp, hs, dp, b, 2 * dp, 2 * hs, dp, dleft};
    p[1] = {u, dp, hs, dp, b ? b + dp : b, 2 * dp, 2 * hs, dp, dright};
  }
};
}  // namespace
}  // namespace gpa

extern "C" int64_t gpa_quad_grad_partials(const gpa_quad_problem* problem) {
  using namespace gpa;
  if (check_quad(problem)) return -1;
  const QuadProducts q(*problem, nullptr, nullptr, nullptr, nullptr);
  return tn_partials(q.p, 2, problem->heads, problem->rows);
}

extern "C" int gpa_quad_weight_grads(const gpa_quad_problem* problem, const void* u, const void* dab, float* partials,
                                     float* dleft, float* dright, hipStream_t stream) {
  using namespace gpa;
  if (int rc = check_quad(problem)) return rc;
  if (problem->dtype != GPA_DTYPE_BF16) return fail(GPA_HIP_EUNSUPPORTED, "quad weight grads: bf16 only");
  if (!u || !dab || !partials || !dleft || !dright)
    return fail(GPA_HIP_EINVAL, "quad weight grads: u, dab, partials, dleft and dright required");
  for (const void* x : {u, dab, (const void*)partials, (const void*)dleft, (const void*)dright})
    if (reinterpret_cast<uintptr_t>(x) % 16) partials = nullptr;  // the workspace's passes take whole 16-byte pieces
  const QuadProducts q(*problem, u, dab, dleft, dright);
  if (int rc = launch_tn_products(q.p, 2, problem->heads, problem->rows, true, stream, partials)) return rc;
  return check_launch("gpa_quad_weight_grads");
}
