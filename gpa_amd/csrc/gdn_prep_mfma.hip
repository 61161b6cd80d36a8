// Chunk preparation of the GDN scan on MFMA: one block per (chunk, stream), 8
// waves (gdn_prep_mfma, gdn_prep_frag).  Per chunk of positions t, u < 64:
//   G     in-chunk cumulative log decay (a wave scan of g)
//   Kn,Qn x/|x| rounded to the activation type, on the bf16 MFMA path also as
//         fragments
//   A     strictly lower b_t e^{G_t-G_u} Kn_t . Kn_u          (K Kn^T on MFMA)
//   T     (I + A)^-1 (unit_lower_inverse)
//   W     T diag(b e^G) Kn   (bf16 hi/lo fragments, or fp32 rows)
//   U     T diag(b) V        (fp32, value-major or in fragment order)
// with the layouts of include/gpa_hip.h.  Reference: the WY form of the
// chunked gated delta rule that src/gpa/ops.py:49-85 runs per token.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "mfma_tiles.h"

namespace gpa {

constexpr int PREP_WAVES = 8, PREP_NT = 64 * PREP_WAVES;

constexpr int PREP_LT = R + 4;  // row pitch of A and T in LDS

// T = (I + A)^-1 of a strictly lower 64 x 64 A (zeros on and above the diagonal
// of its 16 x 16 diagonal blocks; the blocks above them are not read), by every
// thread of the workgroup: t_s starts as zeros, A and T rows PREP_LT apart.
// Wave 0 inverts the four diagonal blocks by forward substitution, a column
// per lane, in registers; then block rows i = 1..3 of 16: T_ij = -T_ii sum_{j<=m<i}
// A_im T_mj on the fp32 MFMA, block column j by wave j: its sums and tiles go from the
// accumulators to the next product's B operand in registers (acc_inorder), so that the
// waves do not meet in between.  Every sum runs over the
// rows in order: for nearly parallel keys, whose terms cancel from row to row, any
// other order adds large partial sums (an error of 1.5e-7 of T's norm at b = 0.88
// in the order in which mma16 takes four adjacent rows a lane, 3e-8 in order).
// Bound: the latency of 16 substitution steps and of wave 0's 36 MFMAs.  Against forward substitution
// through LDS with run-time trip counts and scalar block products (the same sums),
// the prep of 32 streams x 64 chunks of 128 keys takes 27 us less (of 170).
__device__ __forceinline__ void unit_lower_inverse(const float* a_s, float* t_s, int wave, int lane) {
  constexpr int LT = PREP_LT;
  const int c = lane & 15, q = lane >> 4;
  if (wave == 0) {
    const float* ab = a_s + 16 * q * (LT + 1);
    float x[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      float acc = t == c ? 1.f : 0.f;
#pragma unroll
      for (int g = 0; 4 * g < t; ++g) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(ab + t * LT + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (4 * g + e < t) acc -= a[e] * x[4 * g + e];
      }
      x[t] = acc;
    }
#pragma unroll
    for (int t = 0; t < 16; ++t) t_s[(16 * q + t) * LT + 16 * q + c] = x[t];
  }
  lds_barrier();
  if (wave < 3) {  // block column j = wave, whose tiles stay in registers as B operands
    const int j = wave;
    f32x4 tj[3];
#pragma unroll
    for (int m = 0; m < 3; ++m)
      if (m == j) tj[m] = ld_x_inorder(t_s, LT, 16 * j + c, 16 * j, q);
#pragma unroll
    for (int i = 1; i < 4; ++i) {
      if (i <= j) continue;
      f32x4 x = {0.f, 0.f, 0.f, 0.f}, y = x;
#pragma unroll
      for (int m = 0; m < i; ++m)
        if (m >= j) mma16(x, ld_c_inorder(a_s, LT, 16 * i + c, 16 * m, q), tj[m]);
      mma16(y, ld_c_inorder(t_s, LT, 16 * i + c, 16 * i, q), acc_inorder(x));
#pragma unroll
      for (int e = 0; e < 4; ++e) t_s[(16 * i + 4 * q + e) * LT + 16 * j + c] = -y[e];
      if (i < 3) tj[i] = acc_inorder(-y);
    }
  }
  lds_barrier();
}

// gdn_prep_mfma: float32, and bf16 with K not a multiple of 16.  LDS plan
// (floats): one region holds Kn rows, then the b-scaled V slices; T; A (until
// T is done); per-row scalars.  Up to 128 keys this is under 80 KB, so two
// workgroups share a compute unit.
template <int KM>
struct PrepLayout {
  static constexpr int LK = KM + 4, LT = PREP_LT, VC = 128, LV = VC + 4;
  static constexpr int BIG = R * LK > R * LV ? R * LK : R * LV;
  static constexpr int KN_OFF = 0, T_OFF = BIG, A_OFF = T_OFF + R * LT;
  static constexpr int SC_OFF = A_OFF + R * LT;
  static constexpr int TOTAL = SC_OFF + 4 * R;
  static constexpr size_t BYTES = sizeof(float) * TOTAL;
};

template <typename E, int KM>
__global__ __launch_bounds__(PREP_NT, 1) void gdn_prep_mfma(gpa_gdn_problem p, gpa_gdn_saved sv, int nch) {
  using L = PrepLayout<KM>;
  constexpr int LK = L::LK, LT = L::LT, VC = L::VC, LV = L::LV, NW = PREP_WAVES, NTH = PREP_NT;
  constexpr int KT = KM / 32, NTW = KT >= 4 ? KT / 4 : 1;
  extern __shared__ __align__(16) float smem[];
  float* kn_s = smem + L::KN_OFF;  // [R][LK] Kn (rounded), then b V slices [R][LV]
  float* v_s = kn_s;
  float* t_s = smem + L::T_OFF;    // [R][LT] T
  float* a_s = smem + L::A_OFF;    // [R][LT] A
  float* gam_s = smem + L::SC_OFF;
  float* bet_s = gam_s + R;
  float* sc_s = bet_s + R;  // b e^G
  int* tok_s = reinterpret_cast<int*>(sc_s + R);

  const int n = blockIdx.x, s = blockIdx.y, b = s / p.heads, h = s % p.heads;
  const int K = p.kdim, V = p.vdim, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 31, hh = lane >> 5;
  const bool has_q = p.q.ptr != nullptr;

  // ---- gates: G by a wave-wide inclusive scan (wave 0).
  if (wave == 0) {
    const int tok = token_at(p, n, lane), tt = tok >= 0 ? tok : 0;
    float g = scalar_load(p.g, b, h, tt), be = scalar_load(p.beta, b, h, tt);
    g = tok >= 0 ? g : 0.f;
    be = tok >= 0 ? be : 0.f;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float y = __shfl_up(g, off);
      if (lane >= off) g += y;
    }
    gam_s[lane] = g;
    bet_s[lane] = be;
    sc_s[lane] = be * __expf(g);
    tok_s[lane] = tok;
    sv.gam[rows_off(s, n, nch, 0, 1) + lane] = g;
    sv.beta[rows_off(s, n, nch, 0, 1) + lane] = be;
  }
  // T starts as zeros (its upper blocks stay so).
  for (int i = tid; i < R * LT; i += NTH) t_s[i] = 0.f;

  // ---- normalise keys and queries: wave w owns rows w, w + 8, ...; every
  // load is issued (at a clamped address) before the first use.
  {
    constexpr int NI = KM / 64, NR = R / NW;
    const gpa_operand& qsrc = has_q ? p.q : p.k;
    float xk[NR][NI], xq[NR][NI];
#pragma unroll
    for (int j = 0; j < NR; ++j) {
      const int tok = token_at(p, n, wave + NW * j), tt = tok >= 0 ? tok : 0;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int d = lane + 64 * i, dd = d < K ? d : 0;
        xk[j][i] = op_load<E>(p.k, b, h, tt, dd);
        xq[j][i] = op_load<E>(qsrc, b, h, tt, dd);
      }
    }
#pragma unroll
    for (int j = 0; j < NR; ++j) {
      const int r = wave + NW * j, tok = token_at(p, n, r);
      float sk = 0.f, sq = 0.f;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const bool ok = tok >= 0 && lane + 64 * i < K;
        xk[j][i] = ok ? xk[j][i] : 0.f;
        xq[j][i] = (ok && has_q) ? xq[j][i] : 0.f;
        sk += xk[j][i] * xk[j][i];
        sq += xq[j][i] * xq[j][i];
      }
      const float dk = fmaxf(sqrtf(sum64(sk)), 1e-6f), dq = fmaxf(sqrtf(sum64(sq)), 1e-6f);
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int d = lane + 64 * i;
        const float yk = round_as<E>(xk[j][i] / dk);
        kn_s[r * LK + d] = yk;
        if (d < K) sv.kn[rows_off(s, n, nch, r, K) + d] = yk;
        if (has_q && d < K) sv.qn[rows_off(s, n, nch, r, K) + d] = round_as<E>(xq[j][i] / dq);
      }
    }
  }
  __syncthreads();

  // ---- A = strictly lower b_t e^{G_t-G_u} Kn Kn^T: waves 0-3, one 32x32 tile each.
  if (wave < 4) {
    const int rr = wave >> 1, ru = wave & 1;
    f32x16 acc = {};
    if (std::is_same<E, bf16_t>::value) {
#pragma unroll 4
      for (int g = 0; g < KM / 16; ++g) {
        const int c0 = 16 * g + 8 * hh;
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pack8(kn_s + (32 * rr + li) * LK + c0),
                                                       pack8(kn_s + (32 * ru + li) * LK + c0), acc, 0, 0, 0);
      }
    } else {
#pragma unroll 4
      for (int g = 0; g < KM / 8; ++g) {
        const int c0 = 8 * g + 4 * hh;
        mma8(acc, ld_c(kn_s, LK, 32 * rr + li, c0), ld_c(kn_s, LK, 32 * ru + li, c0));
      }
    }
    const int u = 32 * ru + li;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int t = 32 * rr + acc_row(r, hh);
      a_s[t * LT + u] = (u < t) ? bet_s[t] * __expf(gam_s[t] - gam_s[u]) * acc[r] : 0.f;
    }
  }
  __syncthreads();

  unit_lower_inverse(a_s, t_s, wave, lane);
  {
    float* tri = sv.tri + rows_off(s, n, nch, 0, R);
    for (int i = tid; i < R * R / 4; i += NTH) {
      const int t = i / (R / 4), c = 4 * (i % (R / 4));
      *reinterpret_cast<f32x4*>(tri + t * R + c) = *reinterpret_cast<const f32x4*>(t_s + t * LT + c);
    }
  }

  // ---- W = T diag(b e^G) Kn.  Waves below 2 KT own NTW tiles (32 rt, 32 kt).
  const bool own = wave < 2 * KT;
  const int kt = own ? (NTW == 2 ? wave : wave % KT) : 0;
  auto tile_rt = [&](int m) { return NTW == 2 ? m : (own ? wave / KT : 0); };
  f32x16 acc[NTW];
#pragma unroll
  for (int m = 0; m < NTW; ++m) acc[m] = f32x16{};
  if (own) {
#pragma unroll 4
    for (int g = 0; g < R / 8; ++g) {
      const int c0 = 8 * g + 4 * hh;
      const f32x4 bk = ld_x(kn_s, LK, 32 * kt + li, c0);
      const f32x4 sc = *reinterpret_cast<const f32x4*>(sc_s + c0);
#pragma unroll
      for (int m = 0; m < NTW; ++m) mma8(acc[m], ld_c(t_s, LT, 32 * tile_rt(m) + li, c0) * sc, bk);
    }
  }
  if (own) {
    const int k = 32 * kt + li;
    if (k < K) {
#pragma unroll
      for (int m = 0; m < NTW; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) sv.w[rows_off(s, n, nch, 32 * tile_rt(m) + acc_row(r, hh), K) + k] = acc[m][r];
    }
  }

  // ---- U = T diag(b) V in slices of 128 values; every wave owns one 32x32 tile.
  float* um = sv.u + vc_off(s, n, nch, V);
  const int urt = wave >> 2, uvt = wave & 3;
  for (int v0 = 0; v0 < V; v0 += VC) {
    __syncthreads();  // Kn (or the previous slice) is done with
    {
      constexpr int PER = R * VC / PREP_NT;
      float x[PER];
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int idx = tid + NTH * i, r = idx / VC, c = idx % VC, v = v0 + c;
        const int tok = tok_s[r];
        const bool ok = tok >= 0 && v < V;
        x[i] = op_load<E>(p.v, b, h, ok ? tok : 0, ok ? v : 0);
      }
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int idx = tid + NTH * i, r = idx / VC, c = idx % VC, v = v0 + c;
        const bool ok = tok_s[r] >= 0 && v < V;
        v_s[r * LV + c] = ok ? bet_s[r] * x[i] : 0.f;
      }
    }
    __syncthreads();
    f32x16 acc = {};
#pragma unroll 4
    for (int g = 0; g < R / 8; ++g) {
      const int c0 = 8 * g + 4 * hh;
      mma8(acc, ld_c(t_s, LT, 32 * urt + li, c0), ld_x(v_s, LV, 32 * uvt + li, c0));
    }
    const int v = v0 + 32 * uvt + li;
    if (v < V) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4*>(um + (int64_t)v * R + 32 * urt + 8 * q + 4 * hh) =
            f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    }
  }
}

// ---------------------------------------------------------------------------
// Lanes l/8 = 0..7 of one l%8 hold the rows of an 8 x 8 bf16 matrix; returns
// its columns the same way.  Bits 2 and 1 of the row trade places with the
// dword index, bit 0 with the half of a dword.
__device__ __forceinline__ uint4 transpose8(uint4 v, int lane) {
  swap_halves(v.x, v.z);
  swap_halves(v.y, v.w);
  swap_quarters(v.x, v.y);
  swap_quarters(v.z, v.w);
  const uint32_t sel = lane & 8 ? 0x07060302u : 0x01000504u;
  uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t other = __builtin_amdgcn_mov_dpp(d[i], DPP_XOR8, 0xf, 0xf, false);
    d[i] = __builtin_amdgcn_perm(d[i], other, sel);
  }
  return make_uint4(d[0], d[1], d[2], d[3]);
}

__device__ __forceinline__ bf16x8 as_bf16x8(uint4 v) {
  bf16x8 r;
  __builtin_memcpy(&r, &v, 16);
  return r;
}

// gdn_prep_frag: the same chunk preparation for the bf16 MFMA path (bf16
// activations, K a multiple of 16), built around the fragments it writes.  Wave w
// holds rows 8 w .. 8 w + 7; lane (r = l/8, l%8) holds 8-key pieces (or 8-value
// ones) of row 8 w + r, read in 16-byte loads that are all issued first.  A
// normalised key piece is a krow piece as it stands; the 8 x 8 in-wave
// transpose (transpose8) of a piece is a kcol / qcol piece, and of a value
// piece the B operand of U.  krow, then kcol pass through LDS (same place) as
// the operands of A and W.  W and U are fp32 products, summed as in gdn_prep_mfma
// (mma8), and the row norms as there, so that its results keep the bits that
// element-wise loads and LDS rows gave; a tile of W gives both orders of its
// fragments, the second through an in-wave transpose.  The barriers order LDS
// alone, so stores drain behind the later phases.  52 KB of LDS at 128 keys
// (three workgroups per compute unit), 68 KB at 256 (two).
// Bound: HBM.  At 128 x 128 a chunk reads 48 KB and writes 176 KB: 32 streams x
// 64 chunks take 92-97 us, 5.0-5.2 TB/s; the same arithmetic with the rows and fragments
// through float32 LDS rows, element-wise loads and transposed stores took 170 us.
// K = 256, 16 streams x 32 chunks: 92 -> 43 us; one workgroup alone: 34 -> 20 us.
// (T split exactly in three bf16 parts, for the bf16 MFMA, is faster by 2, 4 and 3 us
// at the same error, but its sums round otherwise, and each bf16 rounding that flips
// travels through the layers: 4e-4 of a layer's output, 5e-3 of the LM layer's.)
template <int KM>
struct PrepFragLayout {
  static constexpr int FRAG = (KM < 128 ? 128 : KM) * R * 2;  // bytes of the krow / kcol fragments
  static constexpr int T_OFF = FRAG, A_OFF = T_OFF + 4 * R * PREP_LT, SC_OFF = A_OFF + 4 * R * PREP_LT;
  static constexpr size_t BYTES = SC_OFF + 4 * 3 * R;
};

// VEC: every row of q, k and v starts on a 16-byte boundary and V % 8 == 0.
template <int KM, bool VEC>
__global__ __launch_bounds__(PREP_NT, KM <= 128 ? 6 : 4) void gdn_prep_frag(gpa_gdn_problem p, gpa_gdn_saved sv, int nch) {
  using L = PrepFragLayout<KM>;
  constexpr int LT = PREP_LT, NP = KM / 64, VC = 128, NM = KM >= 256 ? KM / 128 : 1;
  extern __shared__ __align__(16) unsigned char smem_b[];
  uint4* frag_s = reinterpret_cast<uint4*>(smem_b);           // krow pieces, then kcol pieces
  float* t_s = reinterpret_cast<float*>(smem_b + L::T_OFF);   // [R][LT] T
  float* a_s = reinterpret_cast<float*>(smem_b + L::A_OFF);   // [R][LT] A, then the value pieces of a slice
  uint4* vf_s = reinterpret_cast<uint4*>(smem_b + L::A_OFF);
  float* gam_s = reinterpret_cast<float*>(smem_b + L::SC_OFF);
  float* bet_s = gam_s + R;
  float* sc_s = bet_s + R;  // b e^G

  const int n = blockIdx.x, s = blockIdx.y, b = s / p.heads, h = s % p.heads;
  const int K = p.kdim, V = p.vdim, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, hh = lane >> 5, r8 = lane >> 3, pc = lane & 7;
  const int K16 = K / 16, RB = (K + 31) / 32;
  const int64_t chunk_id = (int64_t)s * nch + n;
  const bool has_q = p.q.ptr != nullptr, rows16 = qk_rows_bf16(p);
  const int row = 8 * wave + r8, tok = token_at(p, n, row);

  // Eight elements of this lane's row from column d (clamped), zeros outside.
  auto load8 = [&](const gpa_operand& o, int d, int width) {
    const uint16_t* src = reinterpret_cast<const uint16_t*>(o.ptr) + op_base(o, b, h) + (int64_t)(tok >= 0 ? tok : 0) * o.st;
    if (VEC) return *reinterpret_cast<const uint4*>(src + (d < width ? d : 0));
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int d0 = d + 2 * e, d1 = d0 + 1;
      const uint32_t x = src[d0 < width ? d0 : 0], y = src[d1 < width ? d1 : 0];
      w[e] = (d0 < width ? x : 0u) | (d1 < width ? y << 16 : 0u);
    }
    return make_uint4(w[0], w[1], w[2], w[3]);
  };
  const uint4 zero4 = make_uint4(0u, 0u, 0u, 0u);
  auto keep = [&](uint4 x, int d, int width) { return tok >= 0 && d < width ? x : zero4; };

  uint4 xk[NP], xq[NP], xv[2];
#pragma unroll
  for (int j = 0; j < NP; ++j) xk[j] = load8(p.k, 64 * j + 8 * pc, K);
  if (has_q)
#pragma unroll
    for (int j = 0; j < NP; ++j) xq[j] = load8(p.q, 64 * j + 8 * pc, K);
#pragma unroll
  for (int j = 0; j < 2; ++j) xv[j] = load8(p.v, 64 * j + 8 * pc, V);

  // ---- gates: G by a wave-wide inclusive scan (wave 0).
  if (wave == 0) {
    const int tg = token_at(p, n, lane), tt = tg >= 0 ? tg : 0;
    float g = scalar_load(p.g, b, h, tt), be = scalar_load(p.beta, b, h, tt);
    g = tg >= 0 ? g : 0.f;
    be = tg >= 0 ? be : 0.f;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float y = __shfl_up(g, off);
      if (lane >= off) g += y;
    }
    gam_s[lane] = g;
    bet_s[lane] = be;
    sc_s[lane] = be * __expf(g);
    sv.gam[rows_off(s, n, nch, 0, 1) + lane] = g;
    sv.beta[rows_off(s, n, nch, 0, 1) + lane] = be;
  }
  for (int i = tid; i < R * LT / 4; i += PREP_NT)  // T starts as zeros (its upper blocks stay so)
    *reinterpret_cast<f32x4*>(t_s + 4 * i) = f32x4{0.f, 0.f, 0.f, 0.f};

  // ---- normalise: x / |x| in float32, rounded to bf16.
  auto normalise = [&](uint4 (&x)[NP]) {
    float ss[8] = {};
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      x[j] = keep(x[j], 64 * j + 8 * pc, K);
      const uint32_t w[4] = {x[j].x, x[j].y, x[j].z, x[j].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float lo = bf2_low(w[e]), hi = bf2_high(w[e]);
        ss[2 * e] += lo * lo;
        ss[2 * e + 1] += hi * hi;
      }
    }
    // Keys 64 apart, then 32, 16, .. 1: the tree of sum64 over a key per lane, so that
    // a late read's queries (gdn_prep_q) round alike.  Recursive halving over the row's
    // eight lanes leaves element l%8 in lane l%8.
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool up = pc & 4;
      const float send = up ? ss[i] : ss[i + 4], own = up ? ss[i + 4] : ss[i];
      ss[i] = own + dpp_xor4(send);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const bool up = pc & 2;
      const float send = up ? ss[i] : ss[i + 2], own = up ? ss[i + 2] : ss[i];
      ss[i] = own + dpp<DPP_XOR2>(send);
    }
    const bool up = pc & 1;
    float sum = (up ? ss[1] : ss[0]) + dpp<DPP_XOR1>(up ? ss[0] : ss[1]);
    sum += dpp_xor4(sum);
    sum += dpp<DPP_XOR2>(sum);
    sum += dpp<DPP_XOR1>(sum);
    const float den = fmaxf(sqrtf(sum), 1e-6f);
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      uint32_t w[4] = {x[j].x, x[j].y, x[j].z, x[j].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = bf2_pack(bf2_low(w[e]) / den, bf2_high(w[e]) / den);
      x[j] = make_uint4(w[0], w[1], w[2], w[3]);
    }
  };
  // A normalised piece as saved rows: bf16 where the MFMA read kernels take
  // them, else float32.
  auto put_rows = [&](float* rows, uint4 x, int d) {
    const int64_t at = rows_off(s, n, nch, row, K) + d;
    if (rows16) {
      *reinterpret_cast<uint4*>(reinterpret_cast<bf16_t*>(rows) + at) = x;
    } else {
      const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
      for (int e = 0; e < 2; ++e)
        *reinterpret_cast<f32x4*>(rows + at + 4 * e) = f32x4{bf2_low(w[2 * e]), bf2_high(w[2 * e]),
                                                             bf2_low(w[2 * e + 1]), bf2_high(w[2 * e + 1])};
    }
  };
  // Place of this lane's transposed piece j in a column-fragment buffer.
  auto col_piece = [&](int k) { return ((k >> 5) * 4 + (wave >> 1)) * 64 + (k & 31) + 32 * (wave & 1); };
  normalise(xk);
  {
    uint4* krow = reinterpret_cast<uint4*>(reinterpret_cast<__bf16*>(sv.krow) + chunk_id * frag_row_elems(K, 8));
    uint4* kcol = reinterpret_cast<uint4*>(reinterpret_cast<__bf16*>(sv.kcol) + chunk_id * frag_col_elems(K, 8));
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      const int d = 64 * j + 8 * pc, k = d + r8;
      if (d < K) {
        const int piece = ((row >> 5) * K16 + (d >> 4)) * 64 + (row & 31) + 32 * ((d >> 3) & 1);
        frag_s[piece] = xk[j];
        krow[piece] = xk[j];
        if (!rows16) put_rows(sv.kn, xk[j], d);
      }
      xk[j] = transpose8(xk[j], lane);
      if (k < 32 * RB) kcol[col_piece(k)] = xk[j];
    }
  }
  lds_barrier();
  // ---- A = strictly lower b_t e^{G_t-G_u} Kn Kn^T: waves 0-2, one 32x32 tile each.
  if (wave < 3) {
    const int rr = (wave + 1) >> 1, ru = wave >> 1;  // (0, 0), (1, 0), (1, 1)
    f32x16 acc = {};
#pragma unroll 4
    for (int g = 0; g < K16; ++g)
      mma_bf16(acc, as_bf16x8(frag_s[(rr * K16 + g) * 64 + lane]), as_bf16x8(frag_s[(ru * K16 + g) * 64 + lane]));
    const int u = 32 * ru + li;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int t = 32 * rr + acc_row(r, hh);
      a_s[t * LT + u] = (u < t) ? bet_s[t] * __expf(gam_s[t] - gam_s[u]) * acc[r] : 0.f;
    }
  }
  if (has_q) {
    normalise(xq);
    uint4* qcol = reinterpret_cast<uint4*>(reinterpret_cast<__bf16*>(sv.qcol) + chunk_id * frag_col_elems(K, 8));
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      const int d = 64 * j + 8 * pc, k = d + r8;
      if (d < K) put_rows(sv.qn, xq[j], d);
      xq[j] = transpose8(xq[j], lane);
      if (k < 32 * RB) qcol[col_piece(k)] = xq[j];
    }
  }
  lds_barrier();
#pragma unroll
  for (int j = 0; j < NP; ++j) {
    const int k = 64 * j + 8 * pc + r8;
    if (k < 32 * RB) frag_s[col_piece(k)] = xk[j];
  }
  unit_lower_inverse(a_s, t_s, wave, lane);

  // ---- V pieces of a slice (in A's place), T out, W = T diag(b e^G) Kn.
  auto put_values = [&](int v0) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int d = 64 * j + 8 * pc;
      vf_s[col_piece(d + r8)] = transpose8(keep(xv[j], v0 + d, V), lane);
    }
  };
  put_values(0);
  if (VC < V)
#pragma unroll
    for (int j = 0; j < 2; ++j) xv[j] = load8(p.v, VC + 64 * j + 8 * pc, V);
  {
    float* tri = sv.tri + rows_off(s, n, nch, 0, R);
    for (int i = tid; i < R * R / 4; i += PREP_NT) {
      const int t = i / (R / 4), c = 4 * (i % (R / 4));
      *reinterpret_cast<f32x4*>(tri + t * R + c) = *reinterpret_cast<const f32x4*>(t_s + t * LT + c);
    }
  }
  // Operands of mma8: T rows 32 rt + l%32 and, from column fragments in LDS, keys
  // (values) 32 tile + l%32, both at positions 8 g + 4 (l/32) .. +3.  (Row tile 0 on
  // waves 0-3, which share the SIMDs of waves 4-7: T is lower triangular, and
  // tile 1 has twice the products.)
  const int rt = wave >> 2, w4 = wave & 3, groups = 4 + 4 * rt;
  auto at4 = [&](const float* a, int g) { return *reinterpret_cast<const f32x4*>(a + 8 * g + 4 * hh); };
  auto col4 = [&](const uint4* frag, int tile, int g) {
    const uint2 x = reinterpret_cast<const uint2*>(frag + (tile * 4 + (g >> 1)) * 64 + li + 32 * (g & 1))[hh];
    return f32x4{bf2_low(x.x), bf2_high(x.x), bf2_low(x.y), bf2_high(x.y)};
  };
  const float* t_row = t_s + (32 * rt + li) * LT;
  if (w4 < RB) {
    f32x16 w[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) w[m] = f32x16{};
#pragma unroll 4
    for (int g = 0; g < groups; ++g) {
      const f32x4 t = at4(t_row, g) * at4(sc_s, g);
#pragma unroll
      for (int m = 0; m < NM; ++m)
        if (w4 + 4 * m < RB) mma8(w[m], t, col4(frag_s, w4 + 4 * m, g));
    }
    __bf16* wrow = reinterpret_cast<__bf16*>(sv.wrow) + chunk_id * frag_row_elems(K, 16);
    __bf16* wcol = reinterpret_cast<__bf16*>(sv.wcol) + chunk_id * frag_col_elems(K, 16);
    const int oct = (lane >> 3) & 3;  // this lane's eight keys of the tile, once transposed
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      const int kt = w4 + 4 * m;
      if (kt >= RB) continue;
#pragma unroll
      for (int gp = 0; gp < 2; ++gp) {
        const SplitBf8 x = split_rows(w[m], gp);
        __bf16* col = wcol + (int64_t)(kt * 4 + 2 * rt + gp) * 1024 + lane * 8;
        *reinterpret_cast<bf16x8*>(col) = x.hi;
        *reinterpret_cast<bf16x8*>(col + 512) = x.lo;
        uint4 hi, lo;
        __builtin_memcpy(&hi, &x.hi, 16);
        __builtin_memcpy(&lo, &x.lo, 16);
        hi = transpose8_lanes(hi, lane);
        lo = transpose8_lanes(lo, lane);
        const int ks = 2 * kt + (oct >> 1);
        __bf16* row = wrow + (int64_t)(rt * K16 + ks) * 1024 + (16 * gp + 8 * hh + (lane & 7) + 32 * (oct & 1)) * 8;
        if (ks < K16) {
          *reinterpret_cast<uint4*>(row) = hi;
          *reinterpret_cast<uint4*>(row + 512) = lo;
        }
      }
    }
  }

  // ---- U = T diag(b) V in slices of 128 values; every wave owns one 32x32 tile.
  float* um = sv.u + ufrag_off(s, n, nch, V);
  for (int v0 = 0; v0 < V; v0 += VC) {
    if (v0) {
      lds_barrier();  // every wave is done with the previous slice
      put_values(v0);
      if (v0 + VC < V)
#pragma unroll
        for (int j = 0; j < 2; ++j) xv[j] = load8(p.v, v0 + VC + 64 * j + 8 * pc, V);
    }
    lds_barrier();
    if (v0 + 32 * w4 < V) {
      f32x16 acc = {};
#pragma unroll 4
      for (int g = 0; g < groups; ++g) mma8(acc, at4(t_row, g), at4(bet_s, g) * col4(vf_s, w4, g));
      // Whole 32-column strips, zero past V (the padded strip is read too).
      const bool ok = v0 + 32 * w4 + li < V;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4*>(um + ufrag_idx((v0 >> 5) + w4, rt, q, lane)) =
            ok ? f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]} : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
}

template <int KM>
int launch_prep_frag(const gpa_gdn_problem& p, const gpa_gdn_saved& sv, int nch, hipStream_t st) {
  const bool vec = rows_aligned(p.k) && rows_aligned(p.v) && p.vdim % 8 == 0 && (!p.q.ptr || rows_aligned(p.q));
  const size_t lds = PrepFragLayout<KM>::BYTES;
  const void* fn = vec ? reinterpret_cast<const void*>(gdn_prep_frag<KM, true>)
                       : reinterpret_cast<const void*>(gdn_prep_frag<KM, false>);
  if (lds > 65536 &&
      hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return fail(GPA_HIP_EHIP, "hipFuncSetAttribute(max dynamic LDS) failed");
  const dim3 grid(nch, p.batch * p.heads), block(PREP_NT);
  if (vec) hipLaunchKernelGGL((gdn_prep_frag<KM, true>), grid, block, lds, st, p, sv, nch);
  else hipLaunchKernelGGL((gdn_prep_frag<KM, false>), grid, block, lds, st, p, sv, nch);
  return GPA_HIP_OK;
}

template <typename E, int KM>
int launch_prep(const gpa_gdn_problem& p, const gpa_gdn_saved& sv, int nch, hipStream_t st) {
  if constexpr (std::is_same<E, bf16_t>::value)
    if (p.kdim % 16 == 0) return launch_prep_frag<KM>(p, sv, nch, st);
  const size_t lds = PrepLayout<KM>::BYTES;
  if (lds > 65536 && hipFuncSetAttribute(reinterpret_cast<const void*>(gdn_prep_mfma<E, KM>),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return fail(GPA_HIP_EHIP, "hipFuncSetAttribute(max dynamic LDS) failed");
  hipLaunchKernelGGL((gdn_prep_mfma<E, KM>), dim3(nch, p.batch * p.heads), dim3(PREP_NT), lds, st, p, sv, nch);
  return GPA_HIP_OK;
}

#define GPA_PREP_MFMA(E, KM) \
  template int launch_prep<E, KM>(const gpa_gdn_problem&, const gpa_gdn_saved&, int, hipStream_t);
GPA_PREP_MFMA(float, 64)
GPA_PREP_MFMA(float, 128)
GPA_PREP_MFMA(float, 256)
GPA_PREP_MFMA(bf16_t, 64)
GPA_PREP_MFMA(bf16_t, 128)
GPA_PREP_MFMA(bf16_t, 256)
#undef GPA_PREP_MFMA

}  // namespace gpa
