// Chunk-parallel GDN backward of bf16 scans on the bf16 MFMA path, one block
// per (chunk, stream), 8 waves: the products of gdn_chunk_bwd_mfma.hip, with
// every operand in MFMA fragment form by the time a product reads it.
//
// The value-axis products contract over v, the slow axis of every saved
// value-major buffer, so the 8 contraction values of a lane's operand are 8
// rows of such a buffer at the lane's column: coalesced 4-byte loads.  The
// state S_n and its gradient dS are read by one wave each (wave = 32-key tile,
// both 32-row tiles) and go from global memory to split operands without
// LDS; D, dD and dO, which every wave reads, are split once by the wave that
// loaded them and pass through LDS as fragments (two buffers, one barrier
// per 32 values).  Y = T^T dD stays on fp32 MFMA, one 16 x 16 tile per wave
// with its T operand in registers.  The key-axis and position-axis products
// read the saved krow / kcol / qcol fragments and Qn rows.
//
// Waves (KM <= 128): 0-3 own dQn and the R x R products dP, X (their lower
// tiles, waves 0-2); 4-7 own dKn (D dS^T and Y S^T), and dA, KK (waves 4-6).
// KM = 256: every wave owns all three R x K products of its 32-key tile;
// dP, P on waves 0-2, X, dA, KK on waves 3-5.  Only the lower-triangular tiles
// of the R x R matrices exist: (0,1) is neither computed, written nor read.
// Their fragments, and their transposes', leave the accumulators through one
// half-wave exchange and an in-wave 8 x 8 transpose.
//
// Bound: the HBM traffic it chooses (the saved fragments and rows, states and their
// gradients: 948 MB read and 135 MB written at 32 streams x 64 chunks of 128 x 128,
// about 0.6 GB of them unavoidable), then a workgroup's chain of phases (one workgroup
// of 256 registers per compute unit).  That launch takes 270 us, 4.0 TB/s, 85 % of a
// copy's rate (419 us with operands split by every wave that reads them); 256 x 128,
// 16 streams x 32 chunks: 123 us (235).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "mfma_tiles.h"

namespace gpa {

constexpr int CF_WAVES = 8, CF_NT = 64 * CF_WAVES;

// LDS plan (bytes).  A round's fragments (bf16 elements from a buffer's
// start): D, dD, Y as [2 steps][2 row tiles][hi, lo][64][8], dO as
// [2][2][64][8].  The R x R matrices' fragments take their place after the value
// loop.  The raw key and query rows stay for the normalisation backward, whose
// results take their place and leave in whole rows.
struct ChunkFragLayout {
  static constexpr int D = 0, DD = D + 8 * 512, Y = DD + 8 * 512, DO = Y + 8 * 512, BUF = DO + 4 * 512;
  // split fragments of the R x R matrices, [2 row tiles][4 steps][hi, lo][64][8] each
  static constexpr int MAT = 8 * 1024, X = 0, DQK = MAT, DQKT = 2 * MAT, DKK = 3 * MAT, DKKT = 4 * MAT;
  static constexpr int STAGE = 5 * MAT * 2;
  static_assert(STAGE >= 2 * BUF * 2, "the rounds' fragments share the matrices' place");
  static constexpr int SC_OFF = STAGE, RAW_OFF = SC_OFF + 4 * (13 * R + 4);
  static constexpr size_t bytes(int km) { return RAW_OFF + 2 * 2 * R * (km + 8); }
};

__device__ __forceinline__ bf16x8 frag8(const void* p) {
  const uint4 w = *reinterpret_cast<const uint4*>(p);
  bf16x8 r;
  __builtin_memcpy(&r, &w, 16);
  return r;
}
// Fragment (step, row tile) of a split buffer / of dO.
__device__ __forceinline__ SplitBf8 lds_split(const __bf16* buf, int vs, int rt, int lane) {
  const __bf16* f = buf + (vs * 2 + rt) * 1024 + lane * 8;
  return SplitBf8{frag8(f), frag8(f + 512)};
}
__device__ __forceinline__ bf16x8 lds_exact(const __bf16* buf, int vs, int rt, int lane) {
  return frag8(buf + (vs * 2 + rt) * 512 + lane * 8);
}
__device__ __forceinline__ void put_split(__bf16* frag, int lane, const SplitBf8& x) {
  *reinterpret_cast<bf16x8*>(frag + lane * 8) = x.hi;
  *reinterpret_cast<bf16x8*>(frag + 512 + lane * 8) = x.lo;
}

// HQ: the call has a read gradient.
template <int KM, bool HQ>
__global__ __launch_bounds__(CF_NT, 2) void gdn_chunk_bwd_frag(gpa_gdn_problem p, gpa_gdn_saved sv,
                                                              gpa_gdn_grads gr, int nch) {
  using L = ChunkFragLayout;
  constexpr int NP = KM / 64;
  constexpr bool ALL = KM > 128;           // every wave owns all products of its tile
  constexpr int NTW = KM >= 128 ? 2 : 1;   // 32-row tiles per owning wave
  extern __shared__ __align__(16) unsigned char smem_b[];
  __bf16* stage = reinterpret_cast<__bf16*>(smem_b);
  float* gam_s = reinterpret_cast<float*>(smem_b + L::SC_OFF);
  float* bet_s = gam_s + R;
  float* dgam_s = bet_s + R;
  float* dbet_s = dgam_s + R;
  float* qnrm_s = dbet_s + R;  // |q_t|, |k_t| of the raw rows
  float* knrm_s = qnrm_s + R;
  float* qdot_s = knrm_s + R;  // sum_k x/|x| . dX of the rows
  float* kdot_s = qdot_s + R;
  float* eg_s = kdot_s + R;  // e^{G_t}
  float* ek_s = eg_s + R;    // e^{G_C - G_t}
  float* qrd_s = ek_s + R;   // 1 / max(|q_t|, 1e-6), 1 / max(|k_t|, 1e-6)
  float* krd_s = qrd_s + R;
  int* tok_s = reinterpret_cast<int*>(krd_s + R);  // token of each row (-1: void)
  float* red_s = krd_s + 2 * R;
  constexpr int LR = KM + 8;
  bf16_t* kraw_s = reinterpret_cast<bf16_t*>(smem_b + L::RAW_OFF);  // [R][LR] raw rows, zeros in void rows and past K
  bf16_t* qraw_s = kraw_s + R * LR;

  const int n = blockIdx.x, s = blockIdx.y, b = s / p.heads, h = s % p.heads;
  const int K = p.kdim, V = p.vdim, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, hh = lane >> 5, l16 = lane & 15, q16 = lane >> 4;
  const int K16 = K / 16, RB = (K + 31) / 32;
  const bool rows16 = qk_rows_bf16(p);
  const int64_t chunk_id = (int64_t)s * nch + n;
  const float* st = sv.states + state_off(s, n, nch, K, V);
  const float* dh = gr.dhend + state_off(s, n, nch, K, V);
  const float* dl = sv.delta + vc_off(s, n, nch, V);
  const float* ddl = gr.ddelta + vc_off(s, n, nch, V);
  const float* tri = sv.tri + rows_off(s, n, nch, 0, R);
  const __bf16* krow = reinterpret_cast<const __bf16*>(sv.krow) + chunk_id * frag_row_elems(K, 8);
  const __bf16* kcol = reinterpret_cast<const __bf16*>(sv.kcol) + chunk_id * frag_col_elems(K, 8);
  const __bf16* qcol = reinterpret_cast<const __bf16*>(sv.qcol) + chunk_id * frag_col_elems(K, 8);

  // ---- roles
  const bool grp_q = ALL || wave < 4, grp_k = ALL || wave >= 4;
  const int w4 = wave & 3;
  const int kt = ALL ? wave : (NTW == 2 ? w4 : w4 & 1);  // 32-key tile of the R x K products
  auto tile_rt = [&](int m) { return NTW == 2 ? m : w4 >> 1; };
  const bool own = kt < RB;
  const int k = 32 * kt + li, kc = k < K ? k : 0;
  const int tp = wave;                     // R x R tile of dP, P (waves 0-2)
  const int tx = ALL ? wave - 3 : wave;    // of X
  const int ta = ALL ? wave - 3 : wave - 4;  // of dA, KK
  auto live3 = [](int t) { return t >= 0 && t < 3; };  // tiles (0,0), (1,0), (1,1)
  auto tile_rr = [](int t) { return (t + 1) >> 1; };
  auto tile_ru = [](int t) { return t >> 1; };
  const int yi = wave & 3, yj = wave >> 2;  // Y tile: rows 16 yi .., values 16 yj .. of a round

  // ---- T operand of Y: T[16 g + 4 (l/16) + e][16 yi + l%16]
  f32x4 tT[4];
#pragma unroll
  for (int g = 0; g < 4; ++g)
#pragma unroll
    for (int e = 0; e < 4; ++e) tT[g][e] = tri[(16 * g + 4 * q16 + e) * R + 16 * yi + l16];

  // Loads of a round's shared operands: one D or dD fragment and (waves 0-3) one
  // dO fragment per wave, the dD rows and raw values of the wave's Y tile.
  float rf[8];
  f32x4 ry[4];
  uint4 rdo;
  bf16_t rv[4];
  int tok4[4];
  float bet4[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    tok4[r] = token_at(p, n, 16 * yi + 4 * q16 + r);
    bet4[r] = sv.beta[rows_off(s, n, nch, 16 * yi + 4 * q16 + r, 1)];
  }
  const int tok_do = token_at(p, n, 32 * (wave & 1) + li);
  auto fetch = [&](int v0) {
    {
      const float* src = wave < 4 ? dl : ddl;
      const int v = v0 + 16 * ((wave >> 1) & 1) + 8 * hh, vc = v < V ? v : 0;
#pragma unroll
      for (int e = 0; e < 8; ++e) rf[e] = src[(vc + e) * R + 32 * (wave & 1) + li];
    }
    const int vy = v0 + 16 * yj + l16, vyc = vy < V ? vy : 0;
#pragma unroll
    for (int g = 0; g < 4; ++g) ry[g] = *reinterpret_cast<const f32x4*>(ddl + vyc * R + 16 * g + 4 * q16);
#pragma unroll
    for (int r = 0; r < 4; ++r) rv[r] = op_raw<bf16_t>(p.v, b, h, tok4[r] >= 0 ? tok4[r] : 0, vyc);
    if (HQ) {  // (waves 4-7 load what waves 0-3 do: no branch between the loads)
      const int v = v0 + 16 * ((wave >> 1) & 1) + 8 * hh, vc = v < V ? v : 0;
      rdo = *reinterpret_cast<const uint4*>(reinterpret_cast<const bf16_t*>(gr.dout.ptr) + op_base(gr.dout, b, h) +
                                            (int64_t)(tok_do >= 0 ? tok_do : 0) * gr.dout.st + vc);
    }
  };
  fetch(0);

  // ---- row norms of the raw keys and queries.
  {
    const int row = 8 * wave + (lane >> 3), pc = lane & 7, tok = token_at(p, n, row), tt = tok >= 0 ? tok : 0;
    const gpa_operand& qsrc = HQ ? p.q : p.k;
    uint4 xk[NP], xq[NP];
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      const int d = 64 * j + 8 * pc, dd = d < K ? d : 0;
      xk[j] = *reinterpret_cast<const uint4*>(reinterpret_cast<const bf16_t*>(p.k.ptr) + op_base(p.k, b, h) + (int64_t)tt * p.k.st + dd);
      xq[j] = *reinterpret_cast<const uint4*>(reinterpret_cast<const bf16_t*>(qsrc.ptr) + op_base(qsrc, b, h) + (int64_t)tt * qsrc.st + dd);
    }
    if (tid < R) {
      const float g = sv.gam[rows_off(s, n, nch, 0, 1) + tid], gc = sv.gam[rows_off(s, n, nch, R - 1, 1)];
      gam_s[tid] = g;
      bet_s[tid] = sv.beta[rows_off(s, n, nch, 0, 1) + tid];
      eg_s[tid] = __expf(g);
      ek_s[tid] = __expf(gc - g);
      dgam_s[tid] = dbet_s[tid] = 0.f;
      qdot_s[tid] = kdot_s[tid] = 0.f;
      tok_s[tid] = token_at(p, n, tid);
    }
    if (tid < 4) red_s[tid] = 0.f;
    auto norm = [&](const uint4 (&x)[NP]) {
      float ss = 0.f;
#pragma unroll
      for (int j = 0; j < NP; ++j) {
        const uint32_t w[4] = {x[j].x, x[j].y, x[j].z, x[j].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float lo = bf2_low(w[e]), hi = bf2_high(w[e]);
          ss += lo * lo;
          ss += hi * hi;
        }
      }
      ss += __shfl_xor(ss, 1);
      ss += __shfl_xor(ss, 2);
      ss += __shfl_xor(ss, 4);
      return sqrtf(ss);
    };
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      const int d = 64 * j + 8 * pc;
      const bool ok = tok >= 0 && d < K;
      xk[j] = ok ? xk[j] : make_uint4(0u, 0u, 0u, 0u);
      xq[j] = ok ? xq[j] : make_uint4(0u, 0u, 0u, 0u);
      *reinterpret_cast<uint4*>(kraw_s + row * LR + d) = xk[j];
      if (HQ) *reinterpret_cast<uint4*>(qraw_s + row * LR + d) = xq[j];
    }
    const float nk = norm(xk), nq = HQ ? norm(xq) : 0.f;
    if (pc == 0) {
      knrm_s[row] = nk;
      qnrm_s[row] = nq;
      krd_s[row] = 1.f / fmaxf(nk, 1e-6f);
      qrd_s[row] = 1.f / fmaxf(nq, 1e-6f);
    }
  }
  lds_barrier();

  // ---- value loop.
  // Accumulators: dka, dkw and, in the same registers where a wave owns either
  // half, dq and dp, xx.
  f32x16 acc0[NTW], acc1[2], accq[NTW], accx = {};
#pragma unroll
  for (int m = 0; m < NTW; ++m) acc0[m] = accq[m] = f32x16{};
  acc1[0] = acc1[1] = f32x16{};
  f32x16(&dka)[NTW] = acc0;
  f32x16(&dkw)[2] = acc1;
  f32x16(&dq)[NTW] = ALL ? accq : acc0;
  f32x16 &dp = ALL ? accx : acc1[0], &xx = ALL ? accx : acc1[1];
  float ddot = 0.f;            // this lane's share of <S_n, dS>
  f32x4 dbp = {0.f, 0.f, 0.f, 0.f};  // sum_v V Y of this lane's four rows
  const int nr = (V + 31) / 32;

  // Eight values (rows of a value-major buffer) of this lane's key.
  auto fetch_keys = [&](float (&x)[8], const float* src, int v) {
    const uint32_t at = (uint32_t)((v < V ? v : 0) * K + kc);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = (src + e * K)[at];
  };
  // The loop over rounds of 32 values, one copy per role: the loads of a round
  // are issued a round ahead (the wave's own operands as soon as the products
  // have taken the present ones; at 256 keys, where the registers do not reach,
  // at the round's start), with no branch between them and their use,
  // so that the waits count exactly.
  auto rounds = [&](auto q_role, auto k_role) {
    constexpr bool QR = decltype(q_role)::value, KR = decltype(k_role)::value;
    float rs[2][8], rds[2][8];
    auto fetch_own = [&](int v0, int vs) {
      const int v = v0 + 16 * vs + 8 * hh;
      if (KR || HQ) fetch_keys(rs[vs], st, v);
      if (KR) fetch_keys(rds[vs], dh, v);
    };
    if (!ALL) {
      fetch_own(0, 0);
      fetch_own(0, 1);
    }
    for (int r0 = 0; r0 < nr; ++r0) {
      const int v0 = 32 * r0, vnext = r0 + 1 < nr ? v0 + 32 : v0;
      __bf16* buf = stage + (r0 & 1) * L::BUF;
      if (ALL) {
        fetch_own(v0, 0);
        fetch_own(v0, 1);
      }
      // shared fragments to LDS
      {
        const bool ok = v0 + 16 * ((wave >> 1) & 1) + 8 * hh < V;
#pragma unroll
        for (int e = 0; e < 8; ++e) rf[e] = ok ? rf[e] : 0.f;
        put_split(buf + (QR && (!KR || wave < 4) ? L::D : L::DD) + (wave & 3) * 1024, lane, split_bf8(rf));
        if (HQ && QR && (!KR || wave < 4))
          *reinterpret_cast<uint4*>(buf + L::DO + wave * 512 + lane * 8) =
              ok && tok_do >= 0 ? rdo : make_uint4(0u, 0u, 0u, 0u);
      }
      {
        const int vy = v0 + 16 * yj + l16;
        const bool ok = vy < V;
        f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int g = 0; g < 4; ++g)
          if (g >= yi) mma16(y, tT[g], ok ? ry[g] : f32x4{0.f, 0.f, 0.f, 0.f});
        __bf16* yf = buf + L::Y + (yj * 2 + (yi >> 1)) * 1024 + (16 * (yi & 1) + 4 * q16 + 32 * (l16 >> 3)) * 8 + (l16 & 7);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const __bf16 hi = (__bf16)y[r];
          yf[8 * r] = hi;
          yf[512 + 8 * r] = (__bf16)(y[r] - (float)hi);
          if (tok4[r] >= 0 && ok) {
            reinterpret_cast<bf16_t*>(gr.dv.ptr)[op_base(gr.dv, b, h) + (int64_t)tok4[r] * gr.dv.st + vy] =
                from_f32<bf16_t>(bet4[r] * y[r]);
            dbp[r] += to_f32(rv[r]) * y[r];
          }
        }
      }
      fetch(vnext);
      lds_barrier();
#pragma unroll
      for (int vs = 0; vs < 2; ++vs) {
        const bool ok = v0 + 16 * vs + 8 * hh < V;
        SplitBf8 bs, bds;
        if (KR || HQ) {
#pragma unroll
          for (int e = 0; e < 8; ++e) rs[vs][e] = ok ? rs[vs][e] : 0.f;
          bs = split_bf8(rs[vs]);
        }
        if (KR) {
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            rds[vs][e] = ok ? rds[vs][e] : 0.f;
            ddot += rs[vs][e] * rds[vs][e];
          }
          bds = split_bf8(rds[vs]);
        }
        if (!ALL) fetch_own(vnext, vs);
        if (QR) {
          if (HQ)
#pragma unroll
            for (int m = 0; m < NTW; ++m) mma_exact_split(dq[m], lds_exact(buf + L::DO, vs, tile_rt(m), lane), bs);
          if (live3(tp) && HQ)
            mma_exact_split(dp, lds_exact(buf + L::DO, vs, tile_rr(tp), lane), lds_split(buf + L::D, vs, tile_ru(tp), lane));
          if (live3(tx))
            mma_split(xx, lds_split(buf + L::DD, vs, tile_rr(tx), lane), lds_split(buf + L::D, vs, tile_ru(tx), lane));
        }
        if (KR)
#pragma unroll
          for (int m = 0; m < NTW; ++m) {
            mma_split(dka[m], lds_split(buf + L::D, vs, tile_rt(m), lane), bds);
            mma_split(dkw[m], lds_split(buf + L::Y, vs, tile_rt(m), lane), bs);
          }
      }
    }
  };
  if constexpr (ALL) rounds(std::true_type{}, std::true_type{});
  else if (wave < 4) rounds(std::true_type{}, std::false_type{});
  else rounds(std::false_type{}, std::true_type{});
  // The first global operands of what follows are loaded now: Qn / Kn at the
  // tile's elements and, up to 128 keys, the operands of the R x R products over
  // the keys (P on waves 0-3, KK on waves 4-7).
  uint2 qv[NTW][4], kv[NTW][4];
  auto load_tile = [&](uint2 (&w)[4], const __bf16* col, int rt) {
#pragma unroll
    for (int g = 0; g < 4; ++g)
      w[g] = *reinterpret_cast<const uint2*>(col + (((own ? kt : 0) * 4 + 2 * rt + (g >> 1)) * 64 + li + 32 * (g & 1)) * 8 + 4 * hh);
  };
  constexpr int KG = ALL ? 1 : KM / 16;
  bf16x8 px[KG], py[KG];
  const bool pre = !ALL && (wave >= 4 || (HQ && rows16));
  if (pre) {
    const int t3 = w4 < 3 ? w4 : 2, rr = tile_rr(t3), ru = tile_ru(t3);
    const __bf16* x = wave >= 4 ? krow + (rr * K16 * 64 + lane) * 8
                                : reinterpret_cast<const __bf16*>(sv.qn) + rows_off(s, n, nch, 32 * rr + li, K) + 8 * hh;
    const int step = wave >= 4 ? 512 : 16;
#pragma unroll
    for (int g = 0; g < KG; ++g) {
      const int gg = g < K16 ? g : 0;
      px[g] = frag8(x + gg * step);
      py[g] = frag8(krow + ((ru * K16 + gg) * 64 + lane) * 8);
    }
  }
  if (grp_q && HQ)
#pragma unroll
    for (int m = 0; m < NTW; ++m) load_tile(qv[m], qcol, tile_rt(m));
  if (grp_k)
#pragma unroll
    for (int m = 0; m < NTW; ++m) load_tile(kv[m], kcol, tile_rt(m));
#pragma unroll
  for (int r = 0; r < 4; ++r) {  // sum over the 16 values of a lane group
    float x = dbp[r];
    x += dpp<DPP_XOR8>(x);
    x += dpp<DPP_XOR7>(x);
    x += dpp<DPP_XOR2>(x);
    x += dpp<DPP_XOR1>(x);
    if (l16 == 0) atomicAdd(&dbet_s[16 * yi + 4 * q16 + r], x);
  }
  // (at 64 keys two waves hold the same S and dS columns, one per row tile)
  if (k >= K || (NTW == 1 && tile_rt(0) != 0)) ddot = 0.f;
  if (grp_k) {
    ddot = sum64(ddot);
    if (lane == 0) atomicAdd(&red_s[0], ddot);
  }
  lds_barrier();  // the fragments are done with their place

  // A per-row array at a tile's accumulator rows.
  auto tile_rows = [&](const float* a, int rt, float (&x)[16]) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(a + 32 * rt + 8 * g + 4 * hh);
#pragma unroll
      for (int i = 0; i < 4; ++i) x[4 * g + i] = v[i];
    }
  };
  // Kn or Qn (rounded) at a tile's accumulator elements, from its column fragments.
  auto tile_vals = [&](const uint2 (&w)[4], float (&x)[16]) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      x[4 * g] = bf2_low(w[g].x);
      x[4 * g + 1] = bf2_high(w[g].x);
      x[4 * g + 2] = bf2_low(w[g].y);
      x[4 * g + 3] = bf2_high(w[g].y);
    }
  };
  // Product over the keys of 32 rows by 32 rows, from fragments: four steps' loads at a time.
  auto keys_product = [&](auto row_frag, int ru) {
    f32x16 c = {};
    if (pre) {
#pragma unroll
      for (int g = 0; g < KG; ++g)
        if (g < K16) mma_bf16(c, px[g], py[g]);
      return c;
    }
    for (int g0 = 0; g0 < K16; g0 += 4) {
      bf16x8 x[4], y[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int g = g0 + i < K16 ? g0 + i : g0;
        x[i] = row_frag(g);
        y[i] = frag8(krow + ((ru * K16 + g) * 64 + lane) * 8);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (g0 + i < K16) mma_bf16(c, x[i], y[i]);
    }
    return c;
  };
  // ---- value-axis terms: scale rows, gate gradients, merge the Y term into dKn.
  if (grp_q && own && HQ) {
#pragma unroll
    for (int m = 0; m < NTW; ++m) {
      const int rt = tile_rt(m);
      float x[16];
      float eg[16];
      tile_rows(eg_s, rt, eg);
      tile_vals(qv[m], x);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        dq[m][r] *= eg[r];
        x[r] *= dq[m][r];
      }
      const float sq = tile_row_sum(x, lane);
      if ((lane & 1) == 0) atomicAdd(&dgam_s[32 * rt + acc_row(sum_index(lane), hh)], sq);
    }
  }
  if (grp_k && own) {
    float rk_total = 0.f;
#pragma unroll
    for (int m = 0; m < NTW; ++m) {
      const int rt = tile_rt(m);
      float x[16], pk[16];
      float ek[16], eg[16], be[16];
      tile_rows(ek_s, rt, ek);
      tile_rows(eg_s, rt, eg);
      tile_rows(bet_s, rt, be);
      tile_vals(kv[m], x);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        dka[m][r] *= ek[r];
        pk[r] = x[r] * dka[m][r];
        const float w = -dkw[m][r];
        x[r] *= w;
        dka[m][r] += be[r] * eg[r] * w;
      }
      const float sk = tile_row_sum(pk, lane), sw = tile_row_sum(x, lane);
      if ((lane & 1) == 0) {
        const int t = 32 * rt + acc_row(sum_index(lane), hh);
        const float eg = eg_s[t];
        atomicAdd(&dgam_s[t], bet_s[t] * eg * sw - sk);
        atomicAdd(&dbet_s[t], eg * sw);
        rk_total += sk;
      }
    }
    rk_total = sum64(rk_total);
    if (lane == 0) atomicAdd(&dgam_s[R - 1], rk_total);
  }
  // An R x R tile (rr, ru) into the fragments of its transpose (rows = the tile's
  // columns), which its accumulators hold in order, and of the matrix itself.
  auto put_transposed = [&](int mat, const SplitBf8& x, int gp, int rr, int ru) {
    put_split(stage + mat + (ru * 4 + 2 * rr + gp) * 1024, lane, x);
  };
  auto put_straight = [&](int mat, const SplitBf8& x, int gp, int rr, int ru) {
    const int oct = (lane >> 3) & 3;  // this lane's eight columns of the tile, once transposed
    __bf16* f = stage + mat + (rr * 4 + 2 * ru + (oct >> 1)) * 1024 + (16 * gp + 8 * hh + (lane & 7) + 32 * (oct & 1)) * 8;
    uint4 w;
    __builtin_memcpy(&w, &x.hi, 16);
    *reinterpret_cast<uint4*>(f) = transpose8_lanes(w, lane);
    __builtin_memcpy(&w, &x.lo, 16);
    *reinterpret_cast<uint4*>(f + 512) = transpose8_lanes(w, lane);
  };
  auto mat_frag = [&](int mat, int rt, int ks) {
    const __bf16* f = stage + mat + (rt * 4 + ks) * 1024 + lane * 8;
    return SplitBf8{frag8(f), frag8(f + 512)};
  };
  // ---- X to LDS; dP with P: gate gradients and dQK.
  if (live3(tx))
#pragma unroll
    for (int gp = 0; gp < 2; ++gp) put_transposed(L::X, split_rows(xx, gp), gp, tile_rr(tx), tile_ru(tx));
  if (live3(tp) && HQ) {
    const int rr = tile_rr(tp), ru = tile_ru(tp), u = 32 * ru + li;
    const f32x16 pq = keys_product([&](int g) {
      const int64_t at = rows_off(s, n, nch, 32 * rr + li, K) + 16 * g + 8 * hh;
      return rows16 ? frag8(reinterpret_cast<const bf16_t*>(sv.qn) + at) : pack8(sv.qn + at);
    }, ru);
    float prow[16], pcol = 0.f, gt[16];
    tile_rows(gam_s, rr, gt);
    const float gu = gam_s[u];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const bool live = u <= 32 * rr + acc_row(r, hh);
      const float ex = __expf(live ? gt[r] - gu : 0.f), e = live ? ex : 0.f;
      const float dpv = live ? dp[r] : 0.f;
      const float g = dpv * e * pq[r];
      prow[r] = g;
      pcol += g;
      dp[r] = dpv * e;
    }
#pragma unroll
    for (int gp = 0; gp < 2; ++gp) {
      const SplitBf8 x = split_rows(dp, gp);
      put_transposed(L::DQKT, x, gp, rr, ru);
      put_straight(L::DQK, x, gp, rr, ru);
    }
    const float srow = tile_row_sum(prow, lane);
    if ((lane & 1) == 0) atomicAdd(&dgam_s[32 * rr + acc_row(sum_index(lane), hh)], srow);
    pcol += __shfl_xor(pcol, 32);
    if (hh == 0) atomicAdd(&dgam_s[u], -pcol);
  }
  f32x16 kk = {};
  if (live3(ta))
    kk = keys_product([&](int g) { return frag8(krow + ((tile_rr(ta) * K16 + g) * 64 + lane) * 8); }, tile_ru(ta));
  // Operands of the next two phases: the column fragments of Kn and Qn, T^T rows.
  bf16x8 kf[4], qf[4];
  if (own) {
#pragma unroll
    for (int g = 0; g < 4; ++g) kf[g] = frag8(kcol + ((kt * 4 + g) * 64 + lane) * 8);
    if (grp_k && HQ)
#pragma unroll
      for (int g = 0; g < 4; ++g) qf[g] = frag8(qcol + ((kt * 4 + g) * 64 + lane) * 8);
  }
  float tr[4][8];
  if (live3(ta))
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int e = 0; e < 8; ++e) tr[g][e] = tri[(16 * g + 8 * hh + e) * R + 32 * tile_rr(ta) + li];
  lds_barrier();
  // ---- dA = -(T^T X), strictly lower: b, gate and dKK.
  if (live3(ta)) {
    const int rr = tile_rr(ta), ru = tile_ru(ta), u = 32 * ru + li;
    f32x16 da = {};
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (g < 2 && ta != 0) continue;  // T^T is upper triangular
      mma_split(da, split_bf8(tr[g]), mat_frag(L::X, ru, g));
    }
    float rb[16], rg[16], gcol = 0.f, gt[16], be[16];
    tile_rows(gam_s, rr, gt);
    tile_rows(bet_s, rr, be);
    const float gu = gam_s[u];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const bool live = u < 32 * rr + acc_row(r, hh);  // e^{G_t-G_u} may overflow above the diagonal
      const float dav = live ? -da[r] : 0.f;
      const float ex = __expf(live ? gt[r] - gu : 0.f), e = live ? ex : 0.f;
      const float ekk = e * kk[r];
      rb[r] = dav * ekk;
      const float ga = dav * be[r] * ekk;
      rg[r] = ga;
      gcol += ga;
      da[r] = dav * be[r] * e;
    }
#pragma unroll
    for (int gp = 0; gp < 2; ++gp) {
      const SplitBf8 x = split_rows(da, gp);
      put_transposed(L::DKKT, x, gp, rr, ru);
      put_straight(L::DKK, x, gp, rr, ru);
    }
    const float sb = tile_row_sum(rb, lane), sg = tile_row_sum(rg, lane);
    if ((lane & 1) == 0) {
      const int t = 32 * rr + acc_row(sum_index(lane), hh);
      atomicAdd(&dbet_s[t], sb);
      atomicAdd(&dgam_s[t], sg);
    }
    gcol += __shfl_xor(gcol, 32);
    if (hh == 0) atomicAdd(&dgam_s[u], -gcol);
  }

  // Raw elements of a tile over their row norms (unrounded x/|x|).
  auto raw_over_norm = [&](const bf16_t* raw, const float* rd, int rt, float (&x)[16]) {
    float d[16];
    tile_rows(rd, rt, d);
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] = to_f32(raw[(32 * rt + acc_row(r, hh)) * LR + k]);
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] *= d[r];
  };
  auto add_dots = [&](float (&x)[16], const f32x16& d, float* dot, int rt) {
    float c[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) c[r] = x[r] * d[r];
    const float sum = tile_row_sum(c, lane);
    if ((lane & 1) == 0) atomicAdd(&dot[32 * rt + acc_row(sum_index(lane), hh)], sum);
  };
  // The gradient rows take the raw rows' place in LDS (each lane its own elements) ...
  auto put_grad = [&](bf16_t* rows, const float (&x)[16], const f32x16& d, const float* nrm, const float* dot,
                      const float* rd, int rt) {
    float n16[16], d16[16], r16[16];
    tile_rows(nrm, rt, n16);
    tile_rows(dot, rt, d16);
    tile_rows(rd, rt, r16);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float g = n16[r] > 1e-6f ? d[r] - x[r] * d16[r] : d[r];
      rows[(32 * rt + acc_row(r, hh)) * LR + k] = from_f32<bf16_t>(g * r16[r]);
    }
  };
  // ... and leave in 16-byte pieces, the lanes as in the row norms above.
  auto store_rows = [&](const gpa_operand& dst, const bf16_t* rows) {
    const int row = 8 * wave + (lane >> 3), pc = lane & 7, tok = tok_s[row];
    if (tok < 0) return;
    bf16_t* out = reinterpret_cast<bf16_t*>(dst.ptr) + op_base(dst, b, h) + (int64_t)tok * dst.st;
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      const int d = 64 * j + 8 * pc;
      if (d < K)
        *reinterpret_cast<uint4*>(out + d) = rows ? *reinterpret_cast<const uint4*>(rows + row * LR + d) : make_uint4(0u, 0u, 0u, 0u);
    }
  };
  // ---- dQn += dQK Kn, and its normalisation backward's row sums.
  float xe[NTW][16], qe[NTW][16];
  if (grp_q && own && HQ) {
#pragma unroll
    for (int m = 0; m < NTW; ++m) {
      const int rt = tile_rt(m);
      raw_over_norm(qraw_s, qrd_s, rt, qe[m]);
#pragma unroll
      for (int g = 0; g < 4; ++g)
        if (g < 2 + 2 * rt) mma_split_exact(dq[m], mat_frag(L::DQK, rt, g), kf[g]);
      add_dots(qe[m], dq[m], qdot_s, rt);
    }
  }
  lds_barrier();
  // ---- dKn += dQK^T Qn + (dKK + dKK^T) Kn.
  if (grp_k && own) {
#pragma unroll
    for (int m = 0; m < NTW; ++m) {
      const int rt = tile_rt(m);
      raw_over_norm(kraw_s, krd_s, rt, xe[m]);
#pragma unroll
      for (int g = 0; g < 4; ++g) {  // lower and upper triangular operands
        if (HQ && g >= 2 * rt) mma_split_exact(dka[m], mat_frag(L::DQKT, rt, g), qf[g]);
        if (g < 2 + 2 * rt) mma_split_exact(dka[m], mat_frag(L::DKK, rt, g), kf[g]);
        if (g >= 2 * rt) mma_split_exact(dka[m], mat_frag(L::DKKT, rt, g), kf[g]);
      }
      add_dots(xe[m], dka[m], kdot_s, rt);
    }
  }
  if (grp_q && own && HQ)
#pragma unroll
    for (int m = 0; m < NTW; ++m) put_grad(qraw_s, qe[m], dq[m], qnrm_s, qdot_s, qrd_s, tile_rt(m));
  if (wave == 0) {
    // dg_t = sum_{u >= t} dgam_u: a suffix sum across the wave's lanes
    float acc = dgam_s[lane];
    if (lane == R - 1) acc += __expf(gam_s[R - 1]) * red_s[0];
#pragma unroll
    for (int off = 1; off < R; off <<= 1) {
      const float o = __shfl_down(acc, off, 64);
      if (lane + off < R) acc += o;
    }
    const int tok = tok_s[lane];
    if (tok >= 0) {
      reinterpret_cast<float*>(gr.dg.ptr)[op_base(gr.dg, b, h) + (int64_t)tok * gr.dg.st] = acc;
      reinterpret_cast<float*>(gr.dbeta.ptr)[op_base(gr.dbeta, b, h) + (int64_t)tok * gr.dbeta.st] = dbet_s[lane];
    }
  }
  lds_barrier();
  if (grp_k && own)
#pragma unroll
    for (int m = 0; m < NTW; ++m) put_grad(kraw_s, xe[m], dka[m], knrm_s, kdot_s, krd_s, tile_rt(m));
  if (p.q.ptr && gr.dq.ptr) store_rows(gr.dq, HQ ? qraw_s : nullptr);
  lds_barrier();
  store_rows(gr.dk, kraw_s);
}

template <int KM>
int launch_chunk_bwd_frag(const gpa_gdn_problem& p, const gpa_gdn_saved& sv, const gpa_gdn_grads& gr, int nch,
                          hipStream_t st) {
  const dim3 grid(nch, p.batch * p.heads), block(CF_NT);
  constexpr size_t lds = ChunkFragLayout::bytes(KM);
  const bool hq = p.q.ptr && gr.dout.ptr;
  const void* fn = hq ? reinterpret_cast<const void*>(gdn_chunk_bwd_frag<KM, true>)
                      : reinterpret_cast<const void*>(gdn_chunk_bwd_frag<KM, false>);
  if (lds > 65536 && hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return fail(GPA_HIP_EHIP, "hipFuncSetAttribute(max dynamic LDS) failed");
  if (hq)
    hipLaunchKernelGGL((gdn_chunk_bwd_frag<KM, true>), grid, block, lds, st, p, sv, gr, nch);
  else
    hipLaunchKernelGGL((gdn_chunk_bwd_frag<KM, false>), grid, block, lds, st, p, sv, gr, nch);
  return GPA_HIP_OK;
}
template int launch_chunk_bwd_frag<64>(const gpa_gdn_problem&, const gpa_gdn_saved&, const gpa_gdn_grads&, int, hipStream_t);
template int launch_chunk_bwd_frag<128>(const gpa_gdn_problem&, const gpa_gdn_saved&, const gpa_gdn_grads&, int, hipStream_t);
template int launch_chunk_bwd_frag<256>(const gpa_gdn_problem&, const gpa_gdn_saved&, const gpa_gdn_grads&, int, hipStream_t);

}  // namespace gpa
