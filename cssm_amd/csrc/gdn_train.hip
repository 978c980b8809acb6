// Training kernels of GatedDeltaNetCSSM around its spectral recurrence (gfx950),
// float32, plane-major: the causal short conv + SiLU + input gates of q / k / v and
// their adjoint, the per-pixel norm x output gate and its adjoint, and the adjoint of
// the spectral L2 norm.  The reference takes these gradients with jax.value_and_grad
// (main.py:283) through cssm.py:4763-4859, 4890-4897 and 5026-5141.
// Each is one pass over its planes where a chain of elementwise, padding, slicing and
// reduction launches made ten to thirty (training step of 256 frames x 64 channels of 32 x 32,
// T = 8: 9.1 ms with them, 2.1 ms here).  Bound by HBM, but norm_gate's adjoint by its loads' latency between
// barriers; times at that size (fwd / adjoint):
// qkv_act 86 / 143 us (4.7 / 4.2 TB/s), norm_gate 46 / 180 us (4.4 / 1.9 TB/s), spec_norm_bwd
// 90 us (4.8 TB/s).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "fft_reg.h"
#include "launch.h"

namespace cssm {
namespace {

__device__ __forceinline__ float sigm(float v) { return 1.0f / (1.0f + expf(-v)); }

template <int PX>
__device__ __forceinline__ void ldp(const float* p, float (&v)[PX]) {
  if constexpr (PX == 4) {
    const float4 f = *reinterpret_cast<const float4*>(p);
    v[0] = f.x, v[1] = f.y, v[2] = f.z, v[3] = f.w;
  } else {
    v[0] = *p;
  }
}
template <int PX>
__device__ __forceinline__ void stp(float* p, const float (&v)[PX]) {
  if constexpr (PX == 4)
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  else
    *p = v[0];
}

// the input gate of block blk (1 k, 2 v), channel c, PX pixels at p of frame f:
// mode 1 gates (2, F, HW), 2 (2, F), 3 (F, 2C, HW)
template <int PX>
__device__ __forceinline__ void ld_gate(const QkvActArgs& a, int F, int blk, int c, int f, int p, float (&g)[PX]) {
  if (a.gate_mode == 1) {
    ldp<PX>(a.gates + (size_t(blk - 1) * F + f) * a.HW + p, g);
  } else if (a.gate_mode == 3) {
    ldp<PX>(a.gates + ((size_t(f) * 2 + (blk - 1)) * a.C + c) * a.HW + p, g);
  } else {
    const float v = a.gates[size_t(blk - 1) * F + f];
#pragma unroll
    for (int e = 0; e < PX; ++e) g[e] = v;
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// out = gate * SiLU(o), o_t = b + sum_j w_j raw_{t-KT+1+j} (frames before the first
// are zero); KT = 0: out = gate * raw (the reference applies SiLU only inside the short
// convolution).  One thread per (b, channel of q|k|v, PX pixels) walks the frames.
// ---------------------------------------------------------------------------
template <int KT, int PX>
__global__ void __launch_bounds__(256) qkv_act_fwd(const QkvActArgs a, float* __restrict__ out, long long total) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const int HWq = a.HW / PX, C = a.C, F = a.B * a.T;
  const int p = int(i % HWq) * PX, c3 = int((i / HWq) % (3 * C)), b = int(i / ((long long)HWq * 3 * C));
  const int blk = c3 / C, c = c3 % C;
  constexpr int KW = KT > 0 ? KT : 1;
  float w[KW], bias = 0.0f, R[KW][PX];     // R[k]: frame t - k
#pragma unroll
  for (int j = 0; j < KT; ++j) w[j] = a.sc.w[blk][j * C + c];
  if (KT > 0) bias = a.sc.b[blk][c];
#pragma unroll
  for (int k = 0; k < KW; ++k)
#pragma unroll
    for (int e = 0; e < PX; ++e) R[k][e] = 0.0f;
  for (int t = 0; t < a.T; ++t) {
    const int f = b * a.T + t;
#pragma unroll
    for (int k = KW - 1; k > 0; --k)
#pragma unroll
      for (int e = 0; e < PX; ++e) R[k][e] = R[k - 1][e];
    ldp<PX>(a.raw + size_t(f) * a.raw_fs + size_t(c3) * a.HW + p, R[0]);
    float v[PX];
#pragma unroll
    for (int e = 0; e < PX; ++e) {
      v[e] = R[0][e];
      if (KT > 0) {
        float o = bias;
#pragma unroll
        for (int j = 0; j < KT; ++j) o = fmaf(w[j], R[KT - 1 - j][e], o);
        v[e] = o / (1.0f + expf(-o));
      }
    }
    if (blk > 0 && a.gate_mode) {
      float g[PX];
      ld_gate<PX>(a, F, blk, c, f, p, g);
#pragma unroll
      for (int e = 0; e < PX; ++e) v[e] *= g[e];
    }
    stp<PX>(out + (size_t(f) * 3 * C + c3) * a.HW + p, v);
  }
}

// ---------------------------------------------------------------------------
// Adjoint of qkv_act_fwd.  A wave holds 8 channels x 8 groups of PX pixels (128-byte runs per
// channel) and walks the frames backwards with raw_{t-KT+1..t} and do_{t..t+KT-1} in registers:
//   do_t = dout_t g SiLU'(o_t),  draw_t = sum_l w_{KT-1-l} do_{t+l},
//   dw_{KT-1-l} += do_t raw_{t-l},  db += do_t,  dg_t = dout_t SiLU(o_t)
// dg sums over the channels where they share a gate: the wave's 8 by lane exchange, the groups of 8
// in gpart (2, ceil(C/8), F, HW) for the caller to add (mode 3: written per channel, (F, 2C, HW)).
// A wave takes several pixel groups in turn, so the KT + 2 sums per channel (taps, bias, draw
// itself, which is the projection's bias gradient) leave one partial per (b, blockIdx.x):
// wpart (B, gridDim.x, 3C, KT + 2).  Fixed orders throughout.
// ---------------------------------------------------------------------------
template <int KT, int PX>
__global__ void __launch_bounds__(256) qkv_act_bwd(const QkvActArgs a, const float* __restrict__ dout,
                                                   float* __restrict__ draw, long long draw_fs,
                                                   float* __restrict__ gpart, float* __restrict__ wpart) {
  constexpr int KW = KT > 0 ? KT : 1, NS = KT + 2;
  const int C = a.C, HW = a.HW, T = a.T, F = a.B * T, CGN = (C + 7) / 8;
  const int lane = threadIdx.x & 63, pl = lane & 7, cl = lane >> 3;
  const int grp = int(blockIdx.y) * 4 + (int(threadIdx.x) >> 6), b = blockIdx.z;
  if (grp >= 3 * CGN) return;              // whole waves leave: no barrier below
  const int blk = grp / CGN, cg = grp % CGN, c = cg * 8 + cl;
  const bool cok = c < C;
  const int cs = cok ? c : C - 1, c3 = blk * C + cs;
  float w[KW], bias = 0.0f, acc[NS];
#pragma unroll
  for (int j = 0; j < KT; ++j) w[j] = a.sc.w[blk][j * C + cs];
  if (KT > 0) bias = a.sc.b[blk][cs];
#pragma unroll
  for (int j = 0; j < NS; ++j) acc[j] = 0.0f;
  const bool gated = blk > 0 && a.gate_mode != 0;
  const int nchunk = (HW + 8 * PX - 1) / (8 * PX);
  for (int ch = blockIdx.x; ch < nchunk; ch += gridDim.x) {
    const int p0 = (ch * 8 + pl) * PX;
    const bool ok = cok && p0 < HW;
    const int p = p0 < HW ? p0 : 0;
    const float* rp = a.raw + size_t(b) * T * a.raw_fs + size_t(c3) * HW + p;
    const float* dp = dout + (size_t(b) * T * 3 * C + c3) * HW + p;
    float* wp = draw + size_t(b) * T * draw_fs + size_t(c3) * HW + p;
    float R[KW][PX], D[KW][PX], nr[PX], nd[PX], ng[PX];   // R[k]: raw_{t-k}, D[k]: do_{t+k}
    auto ld_raw = [&](int t, float (&v)[PX]) {
#pragma unroll
      for (int e = 0; e < PX; ++e) v[e] = 0.0f;
      if (t >= 0 && ok) ldp<PX>(rp + size_t(t) * a.raw_fs, v);
    };
    auto ld_next = [&](int t) {       // dout_t and the gates of frame t
#pragma unroll
      for (int e = 0; e < PX; ++e) nd[e] = ng[e] = 0.0f;
      if (t >= 0 && ok) {
        ldp<PX>(dp + size_t(t) * 3 * C * HW, nd);
        if (gated) ld_gate<PX>(a, F, blk, c, b * T + t, p, ng);
      }
    };
#pragma unroll
    for (int k = 0; k < KW; ++k) {
      ld_raw(T - 1 - k, R[k]);
#pragma unroll
      for (int e = 0; e < PX; ++e) D[k][e] = 0.0f;
    }
    ld_raw(T - 1 - KW, nr);
    ld_next(T - 1);
    for (int t = T - 1; t >= 0; --t) {
      float d[PX], g[PX], nr0[PX];
#pragma unroll
      for (int e = 0; e < PX; ++e) d[e] = nd[e], g[e] = ng[e], nr0[e] = nr[e];
      ld_next(t - 1);
      ld_raw(t - KW - 1, nr);
      float dg[PX];
#pragma unroll
      for (int k = KW - 1; k > 0; --k)
#pragma unroll
        for (int e = 0; e < PX; ++e) D[k][e] = D[k - 1][e];
#pragma unroll
      for (int e = 0; e < PX; ++e) {
        float val = R[0][e], slope = 1.0f;
        if (KT > 0) {
          float o = bias;
#pragma unroll
          for (int j = 0; j < KT; ++j) o = fmaf(w[j], R[KT - 1 - j][e], o);
          const float s = sigm(o);
          val = o * s;
          slope = s * fmaf(o, 1.0f - s, 1.0f);
        }
        dg[e] = d[e] * val;
        D[0][e] = (gated ? d[e] * g[e] : d[e]) * slope;
      }
      float dr[PX];
#pragma unroll
      for (int e = 0; e < PX; ++e) {
        dr[e] = KT > 0 ? 0.0f : D[0][e];
#pragma unroll
        for (int l = 0; l < KT; ++l) {
          dr[e] = fmaf(w[KT - 1 - l], D[l][e], dr[e]);
          acc[KT - 1 - l] = fmaf(D[0][e], R[l][e], acc[KT - 1 - l]);
        }
        acc[KT] += D[0][e];
        acc[KT + 1] += dr[e];
      }
      if (ok) stp<PX>(wp + size_t(t) * draw_fs, dr);
      if (gated) {
        const int f = b * T + t;
        if (a.gate_mode == 3) {
          if (ok) stp<PX>(gpart + ((size_t(f) * 2 + (blk - 1)) * C + c) * HW + p, dg);
        } else {
#pragma unroll
          for (int e = 0; e < PX; ++e) {
            dg[e] += __shfl_xor(dg[e], 8, 64);
            dg[e] += __shfl_xor(dg[e], 16, 64);
            dg[e] += __shfl_xor(dg[e], 32, 64);
          }
          if (cl == 0 && p0 < HW) stp<PX>(gpart + ((size_t(blk - 1) * CGN + cg) * F + f) * HW + p, dg);
        }
      }
#pragma unroll
      for (int k = 0; k + 1 < KW; ++k)
#pragma unroll
        for (int e = 0; e < PX; ++e) R[k][e] = R[k + 1][e];
#pragma unroll
      for (int e = 0; e < PX; ++e) R[KW - 1][e] = nr0[e];
    }
  }
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    acc[j] += __shfl_xor(acc[j], 1, 64);
    acc[j] += __shfl_xor(acc[j], 2, 64);
    acc[j] += __shfl_xor(acc[j], 4, 64);
    if (pl == 0 && cok) wpart[((size_t(b) * gridDim.x + blockIdx.x) * 3 * C + c3) * NS + j] = acc[j];
  }
}

// pixel groups per wave so that about 4096 workgroups remain
int qkv_act_bwd_blocks(int B, int C, int HW) {
  const int px = HW % 4 == 0 ? 4 : 1, nchunk = (HW + 8 * px - 1) / (8 * px);
  const long long per = (long long)B * ((3 * ((C + 7) / 8) + 3) / 4);
  const long long want = (4096 + per - 1) / per;
  return int(want < nchunk ? want : nchunk);
}

template <int PX>
static hipError_t run_qkv_act(const QkvActArgs& a, int kt, float* out, const float* dout, float* draw,
                              long long draw_fs, float* gpart, float* wpart, hipStream_t s) {
  const long long total = (long long)a.B * 3 * a.C * (a.HW / PX);
  const dim3 fg(unsigned((total + 255) / 256));
  const dim3 bg(unsigned(qkv_act_bwd_blocks(a.B, a.C, a.HW)), unsigned((3 * ((a.C + 7) / 8) + 3) / 4), unsigned(a.B));
  switch (kt) {
#define CSSM_KT(K)                                                                                                \
  case K:                                                                                                         \
    if (out) hipLaunchKernelGGL((qkv_act_fwd<K, PX>), fg, dim3(256), 0, s, a, out, total);                        \
    else hipLaunchKernelGGL((qkv_act_bwd<K, PX>), bg, dim3(256), 0, s, a, dout, draw, draw_fs, gpart, wpart);     \
    break;
    CSSM_KT(0) CSSM_KT(1) CSSM_KT(2) CSSM_KT(3) CSSM_KT(4) CSSM_KT(5) CSSM_KT(6) CSSM_KT(7) CSSM_KT(8)
#undef CSSM_KT
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_qkv_act_fwd(const QkvActArgs& a, int kt, float* out, hipStream_t s) {
  return a.HW % 4 == 0 ? run_qkv_act<4>(a, kt, out, nullptr, nullptr, 0, nullptr, nullptr, s)
                       : run_qkv_act<1>(a, kt, out, nullptr, nullptr, 0, nullptr, nullptr, s);
}
hipError_t launch_qkv_act_bwd(const QkvActArgs& a, int kt, const float* dout, float* draw, long long draw_fs,
                              float* gpart, float* wpart, hipStream_t s) {
  return a.HW % 4 == 0 ? run_qkv_act<4>(a, kt, nullptr, dout, draw, draw_fs, gpart, wpart, s)
                       : run_qkv_act<1>(a, kt, nullptr, dout, draw, draw_fs, gpart, wpart, s);
}

// ---------------------------------------------------------------------------
// y = (norm(o) scale + shift) act(g) over the channels of each pixel, and its adjoint.  A workgroup
// takes 64 pixels; wave w holds channels w, w + 4, ... of each in registers (KC of them), so o, g
// and dy are read once; the per-pixel sums meet in LDS.  The adjoint walks pixel tiles and keeps its
// channels' scale / shift / gate-bias sums per lane until the end: part (gridDim.x, 3, C).
// norm 0 none, 1 rms, 2 layer; act 1 SiLU, 2 sigmoid.
// ---------------------------------------------------------------------------
struct PixelSums {
  float v[2][4][64];
  // the sum over the four waves of a per-wave value, in wave order; slot k alternates so that one
  // barrier per call is enough
  __device__ __forceinline__ float get(float x, int w, int l, int k) {
    v[k][w][l] = x;
    __syncthreads();
    return ((v[k][0][l] + v[k][1][l]) + v[k][2][l]) + v[k][3][l];
  }
};

template <int KC, bool BWD>
__global__ void __launch_bounds__(256) norm_gate_train(const NormGateArgs a, long long M) {
  __shared__ PixelSums sums;
  const int l = threadIdx.x & 63, w = int(threadIdx.x) >> 6, C = a.C, HW = a.HW;
  const float invC = 1.0f / float(C);
  float sc[KC], bi[KC], as[BWD ? KC : 1], ab[BWD ? KC : 1], ag[BWD ? KC : 1];
#pragma unroll
  for (int k = 0; k < KC; ++k) {
    const int c = w + 4 * k;
    sc[k] = c < C && a.scale ? a.scale[c] : 1.0f;
    bi[k] = c < C && a.shift ? a.shift[c] : 0.0f;
    if (BWD) as[k] = ab[k] = ag[k] = 0.0f;
  }
  for (long long tile = blockIdx.x; tile * 64 < M; tile += gridDim.x) {
    const long long i = tile * 64 + l;
    const bool ok = i < M;
    const long long f = ok ? i / HW : 0;
    const int p = ok ? int(i % HW) : 0;
    const size_t ob = size_t(f) * C * HW + p, gb = size_t(f) * a.g_fs + p, db = size_t(f) * (BWD ? a.dg_fs : 0) + p;
    float o[KC], g[KC], dy[BWD ? KC : 1];
#pragma unroll
    for (int k = 0; k < KC; ++k) {
      const int c = w + 4 * k < C ? w + 4 * k : 0;
      o[k] = a.o[ob + size_t(c) * HW];
      g[k] = a.g[gb + size_t(c) * HW];
      if (BWD) dy[k] = a.dy[ob + size_t(c) * HW];
    }
    float mu = 0.0f, inv = 1.0f;
    if (a.norm == 2) {
      float s = 0.0f;
#pragma unroll
      for (int k = 0; k < KC; ++k) s += w + 4 * k < C ? o[k] : 0.0f;
      mu = sums.get(s, w, l, 0) * invC;
    }
    if (a.norm) {
      float s = 0.0f;
#pragma unroll
      for (int k = 0; k < KC; ++k) s = w + 4 * k < C ? fmaf(o[k] - mu, o[k] - mu, s) : s;
      inv = 1.0f / sqrtf(sums.get(s, w, l, 1) * invC + 1e-6f);
    }
    if constexpr (!BWD) {
#pragma unroll
      for (int k = 0; k < KC; ++k) {
        const int c = w + 4 * k;
        const float s = sigm(g[k]), act = a.act == 1 ? g[k] * s : s;
        if (ok && c < C) a.y[ob + size_t(c) * HW] = fmaf((o[k] - mu) * inv, sc[k], bi[k]) * act;
      }
      if (a.norm == 1) __syncthreads();   // two slots alternate only when both sums are taken
    } else {
      float m1 = 0.0f, m2 = 0.0f;
#pragma unroll
      for (int k = 0; k < KC; ++k) {
        const int c = w + 4 * k;
        const bool use = ok && c < C;
        const float s = sigm(g[k]), act = a.act == 1 ? g[k] * s : s;
        const float slope = a.act == 1 ? s * fmaf(g[k], 1.0f - s, 1.0f) : s * (1.0f - s);
        const float xh = (o[k] - mu) * inv, dn = use ? dy[k] * act : 0.0f;
        const float dg = use ? dy[k] * fmaf(xh, sc[k], bi[k]) * slope : 0.0f;
        if (use) a.dg[db + size_t(c) * HW] = dg;
        as[k] = fmaf(dn, xh, as[k]);
        ab[k] += dn;
        ag[k] += dg;
        dy[k] = dn * sc[k];                 // d xhat
        o[k] = xh;
        m1 += dy[k];
        m2 = fmaf(dy[k], xh, m2);
      }
      if (a.norm) {
        m1 = a.norm == 2 ? sums.get(m1, w, l, 0) * invC : 0.0f;
        if (a.norm == 1) __syncthreads();
        m2 = sums.get(m2, w, l, 1) * invC;
      } else {
        m1 = m2 = 0.0f;
      }
#pragma unroll
      for (int k = 0; k < KC; ++k) {
        const int c = w + 4 * k;
        if (ok && c < C) a.y[ob + size_t(c) * HW] = inv * (dy[k] - m1 - o[k] * m2);
      }
      if (a.norm) __syncthreads();
    }
  }
  if constexpr (BWD) {
#pragma unroll
    for (int k = 0; k < KC; ++k) {
      float v[3] = {as[k], ab[k], ag[k]};
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        for (int off = 32; off > 0; off >>= 1) v[j] += __shfl_xor(v[j], off, 64);
        if (l == 0 && w + 4 * k < C) a.part[(size_t(blockIdx.x) * 3 + j) * C + w + 4 * k] = v[j];
      }
    }
  }
}

bool norm_gate_train_supported(int C) { return C >= 1 && C <= 128; }
// workgroups of the adjoint (its partial sums' first axis)
int norm_gate_blocks(long long M) {
  const long long tiles = (M + 63) / 64;
  return int(tiles < 2048 ? tiles : 2048);
}

hipError_t launch_norm_gate_train(const NormGateArgs& a, long long M, bool bwd, hipStream_t s) {
  if (!norm_gate_train_supported(a.C)) return hipErrorInvalidValue;
  const dim3 grid(unsigned(norm_gate_blocks(M)));
#define CSSM_NG(KC_)                                                                                  \
  if (bwd) hipLaunchKernelGGL((norm_gate_train<KC_, true>), grid, dim3(256), 0, s, a, M);             \
  else hipLaunchKernelGGL((norm_gate_train<KC_, false>), grid, dim3(256), 0, s, a, M);
  if (a.C <= 32) { CSSM_NG(8) }
  else if (a.C <= 64) { CSSM_NG(16) }
  else { CSSM_NG(32) }
#undef CSSM_NG
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Adjoint of the spectral L2 norm of the q and k spectra (cssm.py:4890-4897) followed by the real
// transform's: with n = X r, r = (S + 1e-6)^-1/2, S = sum_bins |X|^2 (norms) and d the gradient of n,
//   dX = (H W / c_v) (r d - r^3 Re(sum_bins conj(d) X) X)
// in place of d (the c_v and H W of rfft2's adjoint, so that irfft2 of the result is the gradient of
// the planes).  One workgroup per plane: the sum, then the update from L2-resident rows.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) spec_norm_bwd(const float2* __restrict__ spec, const float* __restrict__ norms,
                                                     float2* __restrict__ dspec, int C, int H, int W) {
  __shared__ float red[4];
  const int WF = W / 2 + 1, n = H * WF, tid = threadIdx.x;
  const size_t pl = size_t(blockIdx.x / (2 * C)) * 3 * C + blockIdx.x % (2 * C);   // frame, channel of q | k
  const float2* X = spec + pl * n;
  float2* D = dspec + pl * n;
  float s = 0.0f;
  for (int i = tid; i < n; i += 256) {
    const float2 x = X[i], d = D[i];
    s = fmaf(d.x, x.x, fmaf(d.y, x.y, s));
  }
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if ((tid & 63) == 0) red[tid >> 6] = s;
  __syncthreads();
  const float ip = ((red[0] + red[1]) + red[2]) + red[3];
  const float r = 1.0f / sqrtf(norms[pl] + 1e-6f), r3 = r * r * r * ip, hw = float(H * W);
  for (int i = tid; i < n; i += 256) {
    const int v = i % WF;
    const float f = v == 0 || 2 * v == W ? hw : 0.5f * hw;
    const float2 x = X[i], d = D[i];
    D[i] = make_float2(f * fmaf(r, d.x, -r3 * x.x), f * fmaf(r, d.y, -r3 * x.y));
  }
}

hipError_t launch_spec_norm_bwd(const float2* spec, const float* norms, float2* dspec, int F, int C, int H, int W,
                                hipStream_t s) {
  hipLaunchKernelGGL(spec_norm_bwd, dim3(unsigned(2 * C) * unsigned(F)), dim3(256), 0, s, spec, norms, dspec, C, H, W);
  return hipGetLastError();
}

}  // namespace cssm
