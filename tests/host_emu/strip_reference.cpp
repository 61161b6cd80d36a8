// Host build (test infrastructure): the state recurrences of bf16 scans of at
// most 128 keys, element by element in double from the buffers and layouts of
// include/gpa_hip.h.  They stand in for the strip kernels of
// gdn_state_strip.hip, whose global_load_lds inline assembly the emulation does
// not run, so that the kernels before and after them (preparation, output read
// and its gradient, chunk backward) run at these widths.
#include <math.h>

#include <vector>

#include "gdn_common.h"
#include "gdn_strip.h"

namespace gpa {
namespace {

// Element (row t, key k) of a row-fragment block, (key k, position t) of a
// column-fragment block; `planar` blocks hold a 64-lane hi part, then a lo part.
double frag(const __bf16* block, int64_t piece, int lane, int e, bool planar) {
  if (!planar) return (double)(float)block[(piece * 64 + lane) * 8 + e];
  const __bf16* f = block + piece * 1024 + lane * 8 + e;
  return (double)(float)f[0] + (double)(float)f[512];
}
double row_frag(const __bf16* block, int K, int t, int k, bool planar) {
  return frag(block, (t >> 5) * (K / 16) + (k >> 4), (t & 31) + 32 * ((k >> 3) & 1), k & 7, planar);
}
double col_frag(const __bf16* block, int t, int k, bool planar) {
  return frag(block, (k >> 5) * 4 + (t >> 4), (k & 31) + 32 * ((t >> 3) & 1), t & 7, planar);
}
template <typename Pack>
int streams_of(const Pack& pk, int i, int total_wg) {  // one workgroup per stream here
  return (i + 1 < pk.n ? pk.p[i + 1].wg0 : total_wg) - pk.p[i].wg0;
}

void forward(const StripFwdOne& p, int streams) {
  const int K = p.K, V = p.V;
  for (int s = 0; s < streams; ++s) {
    std::vector<double> S(K * V), D(R * V);  // [k][v], [t][v]
    for (int k = 0; k < K; ++k)
      for (int v = 0; v < V; ++v)
        S[k * V + v] = p.s0 ? p.s0[s / p.heads * p.s0_sb + s % p.heads * p.s0_sh + (int64_t)k * V + v] : 0.;
    for (int n = 0; n < p.nch; ++n) {
      const int64_t chunk = (int64_t)s * p.nch + n;
      const __bf16* w = p.wrow + chunk * frag_row_elems(K, 16);
      const __bf16* kc = p.kcol + chunk * frag_col_elems(K, 8);
      const float* g = p.gam + chunk * R;
      for (int k = 0; k < K; ++k)
        for (int v = 0; v < V; ++v) p.states[state_off(s, n, p.nch, K, V) + v * K + k] = (float)S[k * V + v];
      for (int t = 0; t < R; ++t)
        for (int v = 0; v < V; ++v) {
          double d = p.u[ufrag_off(s, n, p.nch, V) + ufrag_elem(v, t)];
          for (int k = 0; k < K; ++k) d -= row_frag(w, K, t, k, true) * S[k * V + v];
          D[t * V + v] = d;
          p.delta[vc_off(s, n, p.nch, V) + v * R + t] = (float)d;
        }
      for (int k = 0; k < K; ++k)
        for (int v = 0; v < V; ++v) {
          double x = exp((double)g[R - 1]) * S[k * V + v];
          for (int t = 0; t < R; ++t) x += col_frag(kc, t, k, false) * exp((double)g[R - 1] - g[t]) * D[t * V + v];
          S[k * V + v] = x;
        }
    }
    for (int i = 0; i < K * V; ++i) p.final_state[(int64_t)s * K * V + i] = (float)S[i];
  }
}

void backward(const StripBwdOne& p, int streams, bool has_q, bool has_inj) {
  const int K = p.K, V = p.V;
  for (int s = 0; s < streams; ++s) {
    std::vector<double> S(K * V), D(R * V);
    for (int i = 0; i < K * V; ++i) S[i] = p.dfinal ? p.dfinal[(int64_t)s * K * V + i] : 0.;
    for (int n = p.nch - 1; n >= 0; --n) {
      const int64_t chunk = (int64_t)s * p.nch + n, uf = ufrag_off(s, n, p.nch, V);
      const __bf16* kr = p.krow + chunk * frag_row_elems(K, 8);
      const __bf16* wc = p.wcol + chunk * frag_col_elems(K, 16);
      const __bf16* qc = has_q ? p.qcol + chunk * frag_col_elems(K, 8) : nullptr;
      const float* g = p.gam + chunk * R;
      const int64_t so = state_off(s, n, p.nch, K, V);
      for (int k = 0; k < K; ++k)
        for (int v = 0; v < V; ++v) p.dhend[so + v * K + k] = (float)S[k * V + v];
      for (int t = 0; t < R; ++t)
        for (int v = 0; v < V; ++v) {
          double d = 0.;
          for (int k = 0; k < K; ++k) d += row_frag(kr, K, t, k, false) * S[k * V + v];
          d = exp((double)g[R - 1] - g[t]) * d + (has_q ? p.dd0[uf + ufrag_elem(v, t)] : 0.);
          D[t * V + v] = d;
          p.ddelta[vc_off(s, n, p.nch, V) + v * R + t] = (float)d;
        }
      for (int k = 0; k < K; ++k)
        for (int v = 0; v < V; ++v) {
          double x = exp((double)g[R - 1]) * S[k * V + v];
          for (int t = 0; t < R; ++t) {
            if (has_q) x += col_frag(qc, t, k, false) * p.o[uf + ufrag_elem(v, t)];
            x -= col_frag(wc, t, k, true) * D[t * V + v];
          }
          S[k * V + v] = x + (has_inj && p.dstates ? p.dstates[so + v * K + k] : 0.);
        }
    }
    for (int i = 0; i < K * V; ++i) p.ds0[(int64_t)s * K * V + i] = (float)S[i];
  }
}

}  // namespace

int strip_wg_per_stream(int, int) { return 1; }
StripFwdOne strip_fwd_one(const gpa_gdn_problem& p, const gpa_gdn_saved& sv, int nch, int wg0, int) {
  return StripFwdOne{p.kdim, p.vdim, p.heads, nch, wg0, 1, p.s0, p.s0_sb, p.s0_sh,
                     static_cast<const __bf16*>(sv.wrow), static_cast<const __bf16*>(sv.kcol), sv.u, sv.gam, sv.delta,
                     sv.states, sv.final};
}
StripBwdOne strip_bwd_one(const gpa_gdn_problem& p, const gpa_gdn_saved& sv, const gpa_gdn_grads& gr, int nch, int wg0,
                          bool has_q, int) {
  return StripBwdOne{p.kdim, p.vdim, p.heads, nch, wg0, 1, gr.dfinal, gr.dstates, gr.dd0, gr.o, gr.ddelta, gr.dhend,
                     gr.ds0, static_cast<const __bf16*>(sv.krow), static_cast<const __bf16*>(sv.wcol),
                     has_q ? static_cast<const __bf16*>(sv.qcol) : nullptr, sv.gam};
}

template <int KM>
int launch_state_fwd_strip(const StripFwdPack& pk, int total_wg, bool, int, hipStream_t) {
  for (int i = 0; i < pk.n; ++i) forward(pk.p[i], streams_of(pk, i, total_wg));
  return 0;
}
template <int KM>
int launch_state_bwd_strip(const StripBwdPack& pk, int total_wg, bool, bool has_q, bool has_inj, int, hipStream_t) {
  for (int i = 0; i < pk.n; ++i) backward(pk.p[i], streams_of(pk, i, total_wg), has_q, has_inj);
  return 0;
}
template int launch_state_fwd_strip<64>(const StripFwdPack&, int, bool, int, hipStream_t);
template int launch_state_fwd_strip<128>(const StripFwdPack&, int, bool, int, hipStream_t);
template int launch_state_bwd_strip<64>(const StripBwdPack&, int, bool, bool, bool, int, hipStream_t);
template int launch_state_bwd_strip<128>(const StripBwdPack&, int, bool, bool, bool, int, hipStream_t);

}  // namespace gpa
