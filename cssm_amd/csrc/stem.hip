// A SimpleCSSM stem layer (simple_cssm.py:266-274): 3 x 3 convolution 'SAME' with bias, and after it the
// activation and the per-pixel LayerNorm ('post' order) or neither ('pre'), then the 2 x 2 maximum.
//
// The convolution is a product of the weights (Co x 9 Ci) with the pixels' neighbourhoods, on the float32
// matrix instruction (32 x 32 x 2: float32 products and sums, chunk by chunk of CK input channels, which at 576
// terms halves the error of one chain): the Co channels are the rows, so a lane holds 16 NM channels of one
// pixel and lane ^ 32 the other half, and bias, activation, LayerNorm and maximum follow in registers.  A
// workgroup of eight waves takes 32 x 16 pixels, a wave two sub-tiles of 16 x 2 (each weight read serves both);
// the tile's CK channels and their weights are staged in LDS at a time, planar with a row pitch of 48 (two rows
// of 16 pixels fall on distinct banks).
//
// Bound by the activation's VALU work in the first layer (18 matrix instructions, 32 softplus a lane) and by the
// matrix instruction in the second (31 of 63 us).  With LayerNorm and softplus, 64 images of 128 x 128 x 3 to
// 32 channels and on from 64 x 64 x 32: 81 and 63 us, where the convolution, bias, activation with norm and
// maximum as separate passes over the unpooled planes, the convolution a library's, took about 470 together.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "launch.h"

namespace cssm {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int TX = 32, TY = 16, SX = TX + 2, SY = TY + 2, PITCH = 48, PL = SY * PITCH;

// log(1 + e^-|v|) = 2 atanh(q), q = t / (2 + t), t = e^-|v| in [0, 1], from atanh's series in z = q^2 <= 1/9 (the
// first term left out is 1.4e-9 of the sum); what q = t rcp(d), d = 2 + t rounded, leaves of the quotient is added
// at the end.  Within one unit in the last place of the true log1p(t); the library's log1pf took 80 of the first
// layer's 132 us.
__device__ __forceinline__ float softplus_tail(float v) {
  const float t = expf(-fabsf(v)), d = 2.0f + t, r = __builtin_amdgcn_rcpf(d);
  const float q = t * r, rest = fmaf(-q, t - (d - 2.0f), fmaf(-q, d, t)) * r, z = q * q;
  float p = 1.0f / 15.0f;
  p = fmaf(p, z, 1.0f / 13.0f);
  p = fmaf(p, z, 1.0f / 11.0f);
  p = fmaf(p, z, 1.0f / 9.0f);
  p = fmaf(p, z, 1.0f / 7.0f);
  p = fmaf(p, z, 1.0f / 5.0f);
  p = fmaf(p, z, 1.0f / 3.0f);
  const float q2 = q + q;
  return q2 + fmaf(q2 * z, p, rest + rest);
}

template <int ACT>
__device__ __forceinline__ float stem_act(float v) {   // as layer_norm_kernel's
  if constexpr (ACT == 1) {
    const float u = 0.7978845608028654f * fmaf(0.044715f * v, v * v, v);
    return 0.5f * v * (1.0f + tanhf(u));
  }
  if constexpr (ACT == 2) return v > 0.0f ? v : (v != v ? v : 0.0f);
  if constexpr (ACT == 3) return fmaxf(v, 0.0f) + softplus_tail(v);
  return v;
}

// the larger, or a NaN of either (as torch's max pooling)
__device__ __forceinline__ float max_nan(float a, float b) { return b > a || b != b ? b : a; }

template <int NM, int CK, bool VEC, int ACT>
__global__ void __launch_bounds__(512, NM == 1 || CK == 4 ? 4 : 2)
stem_conv_kernel(const float* __restrict__ x, int H, int W, int Ci, const float* __restrict__ wt,
                 const float* __restrict__ bias, const float* __restrict__ scale, const float* __restrict__ beta,
                 float eps, int tiles_x, int tiles_y, float* __restrict__ out) {
  constexpr int Co = 32 * NM;
  __shared__ float xs[CK * PL];
  __shared__ __attribute__((aligned(16))) float ws[9 * CK * Co];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int tile = int(blockIdx.x % unsigned(tiles_x * tiles_y));
  const size_t img = blockIdx.x / unsigned(tiles_x * tiles_y);
  const int x0 = (tile % tiles_x) * TX, y0 = (tile / tiles_x) * TY;
  const float* xi = x + img * size_t(H) * W * Ci;
  f32x16 acc[NM][2];
  const int hi = lane >> 5, px = lane & 15, py = (lane >> 4) & 1;
  for (int c0 = 0; c0 < (CK == 4 ? 1 : Ci); c0 += CK) {   // CK = 4: at most 4 channels
    if (c0) __syncthreads();
    for (int p = tid; p < SX * SY; p += 512) {
      const int sy = p / SX, sx = p % SX, gy = y0 + sy - 1, gx = x0 + sx - 1;
      const bool in = gy >= 0 && gy < H && gx >= 0 && gx < W;
      const float* src = xi + (in ? (size_t(gy) * W + gx) * Ci + c0 : 0);
      float v[CK];
      if constexpr (VEC) {                       // Ci a multiple of CK, 16-byte rows
#pragma unroll
        for (int k = 0; k < CK; k += 4) {
          const float4 f = in ? *reinterpret_cast<const float4*>(src + k) : make_float4(0.f, 0.f, 0.f, 0.f);
          v[k] = f.x, v[k + 1] = f.y, v[k + 2] = f.z, v[k + 3] = f.w;
        }
      } else {
#pragma unroll
        for (int k = 0; k < CK; ++k) v[k] = in && c0 + k < Ci ? src[k] : 0.0f;
      }
#pragma unroll
      for (int k = 0; k < CK; ++k) xs[k * PL + sy * PITCH + sx] = v[k];
    }
    for (int e = tid; e < 9 * CK * Co; e += 512) {
      const int co = e % Co, k = (e / Co) % CK, tap = e / (Co * CK);
      ws[e] = c0 + k < Ci ? wt[(size_t(tap) * Ci + c0 + k) * Co + co] : 0.0f;
    }
    __syncthreads();
    f32x16 sum[NM][2];
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < 16; ++i) sum[m][s][i] = 0.0f;
    const float* xb = xs + hi * PL + (2 * w + py) * PITCH + px;
    const float* wb = ws + hi * Co + (lane & 31);
#pragma unroll
    for (int tap = 0; tap < 9; ++tap)
#pragma unroll
      for (int k = 0; k < CK; k += 2) {
        float a[NM], b[2];
#pragma unroll
        for (int m = 0; m < NM; ++m) a[m] = wb[(tap * CK + k) * Co + 32 * m];
#pragma unroll
        for (int s = 0; s < 2; ++s) b[s] = xb[k * PL + (tap / 3) * PITCH + tap % 3 + 16 * s];
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
          for (int s = 0; s < 2; ++s) sum[m][s] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[m], b[s], sum[m][s], 0, 0, 0);
      }
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
      for (int s = 0; s < 2; ++s) acc[m][s] = c0 ? acc[m][s] + sum[m][s] : sum[m][s];
  }
  // element i of acc[m]: channel 32 m + 8 (i / 4) + 4 hi + i % 4 of pixel (px, py)
  const int Ho = (H + 1) / 2, Wo = (W + 1) / 2, gy = y0 + 2 * w + py, quad = (lane & 1) + 2 * py;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int gx = x0 + 16 * s + px;
    const bool in = gy < H && gx < W;
    double sum = 0.0, sq = 0.0;
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 bv = *reinterpret_cast<const float4*>(bias + 32 * m + 8 * g + 4 * hi);
        const float bq[4] = {bv.x, bv.y, bv.z, bv.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float v = stem_act<ACT>(acc[m][s][4 * g + j] + bq[j]);
          acc[m][s][4 * g + j] = v;
          sum += double(v);
          sq = fma(double(v), double(v), sq);
        }
      }
    float mean = 0.0f, rstd = 1.0f;
    if (scale) {
      sum += __shfl_xor(sum, 32, 64);
      sq += __shfl_xor(sq, 32, 64);
      const double mu = sum / Co, var = fmax(sq / Co - mu * mu, 0.0);
      mean = float(mu), rstd = float(1.0 / sqrt(var + double(eps)));
    }
    float* op = out + ((img * Ho + (gy >> 1)) * size_t(Wo) + (gx >> 1)) * Co;
    const bool st = (gy & ~1) < H && (gx & ~1) < W;   // a pooled pixel has at least its first input
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      float4 keep = make_float4(0.f, 0.f, 0.f, 0.f);   // the lane of the four that stores group g
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float r[4];
        float sc[4] = {1.f, 1.f, 1.f, 1.f}, bt[4] = {0.f, 0.f, 0.f, 0.f};
        if (scale) {
          const float4 sv = *reinterpret_cast<const float4*>(scale + 32 * m + 8 * g + 4 * hi);
          const float4 tv = *reinterpret_cast<const float4*>(beta + 32 * m + 8 * g + 4 * hi);
          sc[0] = sv.x, sc[1] = sv.y, sc[2] = sv.z, sc[3] = sv.w;
          bt[0] = tv.x, bt[1] = tv.y, bt[2] = tv.z, bt[3] = tv.w;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float v = acc[m][s][4 * g + j];
          if (scale) v = fmaf((v - mean) * rstd, sc[j], bt[j]);
          v = in ? v : -INFINITY;
          v = max_nan(v, __shfl_xor(v, 1, 64));
          r[j] = max_nan(v, __shfl_xor(v, 16, 64));
        }
        if (quad == g) keep = make_float4(r[0], r[1], r[2], r[3]);
      }
      if (st) *reinterpret_cast<float4*>(op + 32 * m + 8 * quad + 4 * hi) = keep;
    }
  }
}

template <int NM, int ACT>
void run_stem(const float* x, int N, int H, int W, int Ci, const float* wt, const float* bias, const float* scale,
              const float* beta, float eps, float* out, hipStream_t s) {
  const int tx = (W + TX - 1) / TX, ty = (H + TY - 1) / TY;
  const dim3 grid(unsigned((long long)tx * ty * N)), block(512);
  if (Ci <= 4)
    hipLaunchKernelGGL((stem_conv_kernel<NM, 4, false, ACT>), grid, block, 0, s, x, H, W, Ci, wt, bias, scale, beta,
                       eps, tx, ty, out);
  else if (Ci % 8 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0)
    hipLaunchKernelGGL((stem_conv_kernel<NM, 8, true, ACT>), grid, block, 0, s, x, H, W, Ci, wt, bias, scale, beta,
                       eps, tx, ty, out);
  else
    hipLaunchKernelGGL((stem_conv_kernel<NM, 8, false, ACT>), grid, block, 0, s, x, H, W, Ci, wt, bias, scale, beta,
                       eps, tx, ty, out);
}

template <int NM, class... A>
void run_stem_act(int act, A... a) {
  if (act == 0) run_stem<NM, 0>(a...);
  if (act == 1) run_stem<NM, 1>(a...);
  if (act == 2) run_stem<NM, 2>(a...);
  if (act == 3) run_stem<NM, 3>(a...);
}

}  // namespace

bool stem_conv_supported(long long N, int H, int W, int Ci, int Co) {
  return N > 0 && H > 0 && W > 0 && Ci > 0 && (Co == 32 || Co == 64) && H <= 32768 && W <= 32768 &&
         N * ((W + TX - 1) / TX) * ((H + TY - 1) / TY) <= 0x7fffffffLL;
}

hipError_t launch_stem_conv(const float* x, int N, int H, int W, int Ci, int Co, const float* wt, const float* bias,
                            const float* scale, const float* beta, float eps, int act, float* out, hipStream_t s) {
  if (!stem_conv_supported(N, H, W, Ci, Co)) return hipErrorInvalidValue;
  if (Co == 32)
    run_stem_act<1>(act, x, N, H, W, Ci, wt, bias, scale, beta, eps, out, s);
  else
    run_stem_act<2>(act, x, N, H, W, Ci, wt, bias, scale, beta, eps, out, s);
  return hipGetLastError();
}

}  // namespace cssm
