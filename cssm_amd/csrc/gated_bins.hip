// The gated scan's recurrence on spectra in HBM (gfx950): one thread per (b, c,
// frequency bin) walks T frames of rfft2(u), in place:
//   V_t = DB_t U_t, or VF_t where |DB_t U_t| < VF_t;  h_t = Kf E_t h_{t-1} + V_t;
//   spec_t <- C_t h_t
// (cssm.py:559-577 as gated_scan.hip evaluates them; the gate planes' floor term and
// C carry that kernel's factors 2 and c_scale, undone here by exact powers of two).
// Between a batched rfft2 and irfft2 x z this is the fused scan for calls with few
// (b, c) planes: the fused kernel keeps a plane group on one workgroup for all T, so
// with fewer groups than the chip has room for, T steps run one after the other on a
// few CUs; here the transforms of all frames run at once and only this cheap
// recurrence is serial.
// Bound by the latency of its loads at few bins, so U and the gates of the next eight
// frames are in flight while eight are advanced (64-thread workgroups, so that few bins
// still reach every CU).  1024 frames x 256 planes of 16 x 16: transforms and recurrence
// 637 us, the fused kernel 7300 us.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_reg.h"
#include "launch.h"

namespace cssm {

constexpr int kBinsAhead = 8;

// last != nullptr: the final frame stands for reps steps and only its C h is wanted, (B, C, H, WF) in last
// (spec is only read)

__global__ void __launch_bounds__(64) gated_scan_fwd_bins(float2* __restrict__ spec, const float4* __restrict__ gates,
                                                          const float2* __restrict__ khat, float2* __restrict__ state,
                                                          int first, int T, int C, int H, int W, float inv_cs,
                                                          float2* __restrict__ last, int reps) {
  const int WF = W / 2 + 1, HWF = H * WF;
  const int i = int(blockIdx.x) * 64 + int(threadIdx.x), b = blockIdx.y;
  if (i >= C * HWF) return;
  const int c = i / HWF, r = i % HWF, u = r / WF, p = r % WF;
  const float2 kf = khat[size_t(c) * HWF + khat_pos(H, W, u, p)];
  float2* sp = spec + (size_t(b) * T * C + c) * HWF + u * WF + scan_col(H, W, p);
  const size_t fs = size_t(C) * HWF;
  const float4* g = gates + size_t(b) * T * HWF + r;
  float2 h = make_float2(0.f, 0.f);
  if (!first) h = state[size_t(b) * C * HWF + i];
  float2 Un[kBinsAhead];
  float4 Gn[kBinsAhead];
  auto fetch = [&](int t0) {
#pragma unroll
    for (int k = 0; k < kBinsAhead; ++k)
      if (t0 + k < T) {
        Un[k] = sp[size_t(t0 + k) * fs];
        Gn[k] = g[size_t(t0 + k) * HWF];
      }
  };
  fetch(0);
  for (int t0 = 0; t0 < T; t0 += kBinsAhead) {
    float2 U[kBinsAhead];
    float4 G[kBinsAhead];
#pragma unroll
    for (int k = 0; k < kBinsAhead; ++k) {
      U[k] = Un[k];
      G[k] = Gn[k];
    }
    fetch(t0 + kBinsAhead);
#pragma unroll
    for (int k = 0; k < kBinsAhead; ++k) {
      if (t0 + k >= T) break;
      const float vf = 0.5f * G[k].z;
      float2 V = make_float2(U[k].x * G[k].y, U[k].y * G[k].y);
      if (V.x * V.x + V.y * V.y < vf * vf) V = make_float2(vf, 0.f);
      const float2 A = cscale(kf, G[k].x);
      const bool fin = last && t0 + k == T - 1;
      for (int n = fin ? reps : 1; n > 0; --n)
        h = make_float2(fmaf(A.x, h.x, fmaf(-A.y, h.y, V.x)), fmaf(A.x, h.y, fmaf(A.y, h.x, V.y)));
      if (fin) last[(size_t(b) * C + c) * HWF + u * WF + scan_col(H, W, p)] = cscale(h, G[k].w * inv_cs);
      else if (!last) sp[size_t(t0 + k) * fs] = cscale(h, G[k].w * inv_cs);
    }
  }
  if (state) state[size_t(b) * C * HWF + i] = h;
}

hipError_t launch_gated_scan_fwd_bins(float2* spec, const float4* gates, const float2* khat, float2* state, int first,
                                      int B, int T, int C, int H, int W, float c_scale, float2* last, int reps,
                                      hipStream_t s) {
  const long long n = (long long)C * H * (W / 2 + 1);
  hipLaunchKernelGGL(gated_scan_fwd_bins, dim3(unsigned((n + 63) / 64), unsigned(B)), dim3(64), 0, s, spec, gates,
                     khat, state, first, T, C, H, W, 1.0f / c_scale, last, reps);
  return hipGetLastError();
}

}  // namespace cssm
