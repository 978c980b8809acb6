// Caller wiring of CSSMSHViTBlock around the cell: the token-mixer half of
// the block (cssm_shvit.py:86-229): norm1 -> pos_conv -> cell -> frame
// selection -> output activation -> residual, and of the MLP half (:231-266)
// norm2 and the gelu + depthwise convolution between the two products.
//
// Tensors are channels-last (B, T, H, W, C); an image input is (B, 1, H, W, C)
// and is repeated to the cell's T frames on the way out of the pos_conv pass.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <initializer_list>

#include "fft_plane.h"
#include "launch.h"

namespace cssm {
namespace {

__device__ __forceinline__ float ldx(const float* p, size_t i) { return p[i]; }
__device__ __forceinline__ float ldx(const uint16_t* p, size_t i) { return bf16_to_f32(p[i]); }
__device__ __forceinline__ void stx(float* p, size_t i, float v) { p[i] = v; }
__device__ __forceinline__ void stx(uint16_t* p, size_t i, float v) { p[i] = uint16_t(f32_to_bf16(v)); }

// norm1 group of element (b, t, p, c) (p = h W + w) and its element count
//   mode 0 global_layer   (cssm_shvit.py:106-108): b        over T H W C
//   mode 1 temporal_layer (:109-111):              (b, p)   over T C
//   mode 2 layer          (:112-114):              (b, t, p) over C
__device__ __forceinline__ long long norm_group(int mode, int b, int t, int p, int T, int HW) {
  if (mode == 0) return b;
  if (mode == 1) return (long long)b * HW + p;
  return ((long long)b * T + t) * HW + p;
}

}  // namespace

namespace {

// V consecutive elements (V = 4: one vector access, the pointer 4-element aligned) as floats
template <int V>
__device__ __forceinline__ void ldv(const float* p, size_t i, float (&v)[V]) {
  if constexpr (V == 4) {
    const float4 f = *reinterpret_cast<const float4*>(p + i);
    v[0] = f.x, v[1] = f.y, v[2] = f.z, v[3] = f.w;
  } else {
    v[0] = p[i];
  }
}
template <int V>
__device__ __forceinline__ void ldv(const uint16_t* p, size_t i, float (&v)[V]) {
  if constexpr (V == 4) {
    const uint2 u = *reinterpret_cast<const uint2*>(p + i);
    v[0] = bf16_to_f32(u.x & 0xffffu), v[1] = bf16_to_f32(u.x >> 16);
    v[2] = bf16_to_f32(u.y & 0xffffu), v[3] = bf16_to_f32(u.y >> 16);
  } else {
    v[0] = bf16_to_f32(p[i]);
  }
}
template <int V>
__device__ __forceinline__ void stv(float* p, size_t i, const float (&v)[V]) {
  if constexpr (V == 4)
    *reinterpret_cast<float4*>(p + i) = make_float4(v[0], v[1], v[2], v[3]);
  else
    p[i] = v[0];
}
template <int V>
__device__ __forceinline__ void stv(uint16_t* p, size_t i, const float (&v)[V]) {
  if constexpr (V == 4)
    *reinterpret_cast<uint2*>(p + i) =
        make_uint2(f32_to_bf16(v[0]) | (f32_to_bf16(v[1]) << 16), f32_to_bf16(v[2]) | (f32_to_bf16(v[3]) << 16));
  else
    p[i] = uint16_t(f32_to_bf16(v[0]));
}

// sum over the L lanes (a power of two <= 64) that share a group; every lane gets it
__device__ __forceinline__ double lane_sum(double a, int L) {
  for (int off = L / 2; off > 0; off >>= 1) a += __shfl_xor(a, off, 64);
  return a;
}

__device__ __forceinline__ float2 mean_rstd(double a, double q, double n, float eps) {
  const double mean = a / n;
  const double var = fmax(q / n - mean * mean, 0.0);
  return make_float2(float(mean), float(1.0 / sqrt(var + double(eps))));
}

}  // namespace

// stats[g] = (mean, rsqrt(var + eps)) with var = E[x^2] - E[x]^2 (Flax's fast
// variance), sums in double in a fixed order.  mode 0: one 1024-thread workgroup per
// group (few groups of many elements: sixteen waves' 16-byte loads in flight, 64 images of
// 14x14x128 in 5.2 us); modes 1 and 2: one wave per group, four groups per workgroup.
// (One lane adding 64 LDS partials per group, and a scalar load per element, had a CSSM-SHViT
// block's two statistics at 39 us.)
template <int V, class TI>
__global__ void __launch_bounds__(1024)
block_norm_stats_kernel(const TI* __restrict__ x, int T, int HW, int C, int mode, long long groups, float eps,
                        float2* __restrict__ stats) {
  __shared__ double s1[16], s2[16];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  double a = 0.0, q = 0.0;
  auto add = [&](const float (&v)[V]) {
#pragma unroll
    for (int e = 0; e < V; ++e) {
      a += double(v[e]);
      q = fma(double(v[e]), double(v[e]), q);
    }
  };
  if (mode == 0) {
    const long long g = blockIdx.x, n = (long long)T * HW * C;
    const TI* xg = x + g * n;
#pragma unroll 4
    for (long long e = (long long)tid * V; e < n; e += 1024 * V) {
      float v[V];
      ldv<V>(xg, size_t(e), v);
      add(v);
    }
    a = lane_sum(a, 64);
    q = lane_sum(q, 64);
    if (lane == 0) s1[wv] = a, s2[wv] = q;
    __syncthreads();
    if (tid == 0) {
      for (int i = 1; i < 16; ++i) a += s1[i], q += s2[i];
      stats[g] = mean_rstd(a, q, double(n), eps);
    }
    return;
  }
  const long long g = (long long)blockIdx.x * 4 + wv;   // 256 threads
  if (g >= groups) return;
  const int rows = mode == 1 ? T : 1;
  const long long row0 = mode == 1 ? (g / HW) * T * HW + g % HW : g;
  for (int t = 0; t < rows; ++t) {
    const TI* xr = x + (row0 + (long long)t * HW) * C;
    for (int e = lane * V; e < C; e += 64 * V) {
      float v[V];
      ldv<V>(xr, size_t(e), v);
      add(v);
    }
  }
  a = lane_sum(a, 64);
  q = lane_sum(q, 64);
  if (lane == 0) stats[g] = mean_rstd(a, q, double(rows) * C, eps);
}

// out[b, t] = xn + [pos_conv(xn)] for t < T_out, xn = (x[b, t_in] - mean) rstd
// scale + bias with t_in = t (T_in = T_out) or 0 (an image, T_in = 1);
// pos_conv = depthwise 3x3 'SAME' cross-correlation with bias (cssm_shvit.py:
// 122-145), zero padding of xn.  One thread per (input pixel, V channels), V = 4
// with 16-byte accesses where C and the pointers allow; an image's value is computed
// once and stored to its T_out frames, which bounds it (64 images 14x14x128 to 8 frames:
// 17.2 us, 3 TB/s of stores; with the nine taps evaluated again for every frame by element
// loads the block's two calls took 299 us).
template <int V, class TI>
__global__ void __launch_bounds__(256)
block_norm_posconv_kernel(const TI* __restrict__ x, int T_in, int T_out, int H, int W, int C, int mode,
                          const float2* __restrict__ stats, const float* __restrict__ scale,
                          const float* __restrict__ bias, const float* __restrict__ pk, const float* __restrict__ pb,
                          TI* __restrict__ out, long long total) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const int CG = C / V, HW = H * W;
  const int c0 = int(i % CG) * V;
  const long long pix = i / CG;                  // (b, t_in, p)
  const int p = int(pix % HW);
  const long long bt = pix / HW;
  const int ti = int(bt % T_in), b = int(bt / T_in);
  const int h = p / W, w = p % W;
  const TI* xf = x + bt * HW * C;
  float sc[V], bs[V];
  ldv<V>(scale, size_t(c0), sc);
  ldv<V>(bias, size_t(c0), bs);
  // normalised input at (hh, ww), channels c0 ..
  auto xn = [&](int hh, int ww, float (&v)[V]) {
    const float2 st = stats[norm_group(mode, b, ti, hh * W + ww, T_in, HW)];
    ldv<V>(xf, size_t(hh * W + ww) * C + c0, v);
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = fmaf((v[e] - st.x) * st.y, sc[e], bs[e]);
  };
  float acc[V];
  xn(h, w, acc);
  if (pk != nullptr) {
    float pbv[V];
    ldv<V>(pb, size_t(c0), pbv);
#pragma unroll
    for (int e = 0; e < V; ++e) acc[e] += pbv[e];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int hh = h + a - 1;
      if (hh < 0 || hh >= H) continue;
#pragma unroll
      for (int b2 = 0; b2 < 3; ++b2) {
        const int ww = w + b2 - 1;
        if (ww < 0 || ww >= W) continue;
        float kt[V], v[V];
        ldv<V>(pk, size_t((a * 3 + b2) * C + c0), kt);
        xn(hh, ww, v);
#pragma unroll
        for (int e = 0; e < V; ++e) acc[e] = fmaf(kt[e], v[e], acc[e]);
      }
    }
  }
  const size_t o = (size_t(p) * C) + c0;
  if (T_in == T_out) {
    stv<V>(out, size_t(bt) * HW * C + o, acc);
  } else {
    for (int t = 0; t < T_out; ++t) stv<V>(out, (size_t(b) * T_out + t) * HW * C + o, acc);
  }
}

// y = post(LayerNorm(pre(x))) over the last axis of (M, C) rows: statistics as
// block_norm_stats_kernel (double sums, Flax's fast variance) and the normalised value as
// block_norm_posconv_kernel, with the row in registers between them, so x is read once.
// L lanes share a row (64 / L rows per wave), NV vectors of V elements each.  Activations:
// 0 none, 1 gelu (tanh form), 2 relu, 3 softplus.  One read and one write of x, and at few
// channels the activation and the double sums (softplus + norm of 8.4M + 2.1M rows of 32
// channels: 1.1 ms, 2.4 TB/s; activation, statistics and normalisation as three passes 7.1 ms).
// L is chosen for one to two vectors per lane: a row's 16-byte loads then cover whole lines.
__device__ __forceinline__ float ln_act(float v, int act) {
  if (act == 1) {
    const float u = 0.7978845608028654f * fmaf(0.044715f * v, v * v, v);
    return 0.5f * v * (1.0f + tanhf(u));
  }
  if (act == 2) return v > 0.0f ? v : (v != v ? v : 0.0f);
  if (act == 3) return fmaxf(v, 0.0f) + log1pf(expf(-fabsf(v)));
  return v;
}

template <int V, int NV, class TI>
__global__ void __launch_bounds__(256)
layer_norm_kernel(const TI* __restrict__ x, long long M, int C, int L, float eps, const float* __restrict__ scale,
                  const float* __restrict__ bias, int pre, int post, TI* __restrict__ out) {
  const int rpb = 256 / L, lane = threadIdx.x % L;
  const long long row = (long long)blockIdx.x * rpb + threadIdx.x / L;
  const bool live = row < M;
  const TI* xr = x + (live ? row : 0) * C;
  float v[NV][V];
  double a = 0.0, q = 0.0;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int e = (k * L + lane) * V;
    if (live && e < C) ldv<V>(xr, size_t(e), v[k]);
  }
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int e = (k * L + lane) * V;
    if (live && e < C) {
#pragma unroll
      for (int j = 0; j < V; ++j) {
        v[k][j] = ln_act(v[k][j], pre);
        a += double(v[k][j]);
        q = fma(double(v[k][j]), double(v[k][j]), q);
      }
    }
  }
  a = lane_sum(a, L);
  q = lane_sum(q, L);
  if (!live) return;
  const float2 st = mean_rstd(a, q, double(C), eps);
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int e = (k * L + lane) * V;
    if (e >= C) break;
    float sc[V], bs[V];
    ldv<V>(scale, size_t(e), sc);
    ldv<V>(bias, size_t(e), bs);
#pragma unroll
    for (int j = 0; j < V; ++j) v[k][j] = ln_act(fmaf((v[k][j] - st.x) * st.y, sc[j], bs[j]), post);
    stv<V>(out, size_t(row) * C + e, v[k]);
  }
}

// The inside of an MLP with a depthwise convolution (shvit.py:156-182): out = g + conv3x3(g) + bias, g = gelu(x), over
// (N, H, W, C).  A workgroup takes R rows of one image and 32 channels: their gelu values with a row either side go
// to LDS once (as eight 16-byte channel groups a pixel), then each thread, whose channel group and weights are fixed,
// sums nine of them per output.  Rows are the most that fit 64 KB.  One read and one write of x; 64 images of
// 14 x 14 x 512: 18.3 us (2.8 TB/s; the nine LDS reads and the gelu share it), as gelu, convolution and addition 51 us.
constexpr int kMlpPix = 512;   // pixels of 32 channels in LDS

__global__ void __launch_bounds__(256)
mlp_dwconv_kernel(const float* __restrict__ x, int H, int W, int C, int R, int tiles, const float* __restrict__ k3,
                  const float* __restrict__ bias, float* __restrict__ out) {
  extern __shared__ float4 g[];
  const int tid = threadIdx.x, q = tid & 7, c = int(blockIdx.y) * 32 + 4 * q;
  const int y0 = int(blockIdx.x % unsigned(tiles)) * R, rows = min(R, H - y0);
  const size_t base = size_t(blockIdx.x / unsigned(tiles)) * H * W * C + c;
  const int lo = max(y0 - 1, 0), hi = min(y0 + rows + 1, H);   // image rows in LDS
  for (int p = tid >> 3; p < (hi - lo) * W; p += 32) {
    const float4 v = *reinterpret_cast<const float4*>(x + base + size_t(lo * W + p) * C);
    g[p * 8 + q] = make_float4(ln_act(v.x, 1), ln_act(v.y, 1), ln_act(v.z, 1), ln_act(v.w, 1));
  }
  float4 w9[9];
#pragma unroll
  for (int t = 0; t < 9; ++t) w9[t] = *reinterpret_cast<const float4*>(k3 + size_t(t) * C + c);
  const float4 bv = *reinterpret_cast<const float4*>(bias + c);
  __syncthreads();
  for (int p = tid >> 3; p < rows * W; p += 32) {
    const int y = y0 + p / W, xx = p % W;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int t = 0; t < 9; ++t) {
      const int sy = y + t / 3 - 1, sx = xx + t % 3 - 1;
      if (sy < 0 || sy >= H || sx < 0 || sx >= W) continue;
      const float4 v = g[((sy - lo) * W + sx) * 8 + q];
      a.x = fmaf(w9[t].x, v.x, a.x), a.y = fmaf(w9[t].y, v.y, a.y);
      a.z = fmaf(w9[t].z, v.z, a.z), a.w = fmaf(w9[t].w, v.w, a.w);
    }
    const float4 v = g[((y - lo) * W + xx) * 8 + q];
    *reinterpret_cast<float4*>(out + base + size_t(y * W + xx) * C) =
        make_float4(v.x + (a.x + bv.x), v.y + (a.y + bv.y), v.z + (a.z + bv.z), v.w + (a.w + bv.w));
  }
}

// out[b, t] = res[b, tr] + act(y[b, ty]) over (H, W, C): T_out = 1 takes the
// last frame of each (cssm_shvit.py:211, :224), T_out > 1 frame t of both
// (keep_time, :213, :222).  act 0 none, 1 gelu (tanh form, jax.nn.gelu's
// default), 2 silu (:215-218).
template <class TI>
__global__ void __launch_bounds__(256)
block_residual_kernel(const TI* __restrict__ res, int T_res, const TI* __restrict__ y, int T_y, int T_out, int HWC,
                      int act, TI* __restrict__ out, long long total) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const long long e = i % HWC, bt = i / HWC;
  const int t = int(bt % T_out), b = int(bt / T_out);
  const int tr = T_out == 1 ? T_res - 1 : t, ty = T_out == 1 ? T_y - 1 : t;
  float v = ldx(y, size_t(((long long)b * T_y + ty) * HWC + e));
  if (act == 1) {
    const float u = 0.7978845608028654f * fmaf(0.044715f * v, v * v, v);
    v = 0.5f * v * (1.0f + tanhf(u));
  } else if (act == 2) {
    v = v / (1.0f + expf(-v));
  }
  stx(out, size_t(i), ldx(res, size_t(((long long)b * T_res + tr) * HWC + e)) + v);
}

static unsigned blocks_for(long long n, int per) { return unsigned((n + per - 1) / per); }

// 4-element accesses of dtype elements: C a multiple of 4 and every pointer aligned
static bool vec4_ok(int dtype, int C, std::initializer_list<const void*> io, std::initializer_list<const void*> f32s) {
  if (C % 4) return false;
  for (const void* p : io)
    if (reinterpret_cast<uintptr_t>(p) % (dtype == 0 ? 16 : 8)) return false;
  for (const void* p : f32s)
    if (reinterpret_cast<uintptr_t>(p) % 16) return false;
  return true;
}

template <class TI>
static void run_norm_stats(const void* x, int T, int HW, int C, int mode, long long groups, float eps, float2* stats,
                           bool v4, hipStream_t s) {
  const dim3 grid(blocks_for(groups, mode == 0 ? 1 : 4)), block(mode == 0 ? 1024 : 256);
  if (v4)
    hipLaunchKernelGGL((block_norm_stats_kernel<4, TI>), grid, block, 0, s, static_cast<const TI*>(x), T, HW, C, mode,
                       groups, eps, stats);
  else
    hipLaunchKernelGGL((block_norm_stats_kernel<1, TI>), grid, block, 0, s, static_cast<const TI*>(x), T, HW, C, mode,
                       groups, eps, stats);
}

hipError_t launch_block_norm_stats(const void* x, int dtype, int B, int T, int H, int W, int C, int mode, float eps,
                                   float* stats, hipStream_t s) {
  const int HW = H * W;
  const long long groups = mode == 0 ? B : (mode == 1 ? (long long)B * HW : (long long)B * T * HW);
  const bool v4 = vec4_ok(dtype, C, {x}, {});
  if (dtype == 0)
    run_norm_stats<float>(x, T, HW, C, mode, groups, eps, reinterpret_cast<float2*>(stats), v4, s);
  else
    run_norm_stats<uint16_t>(x, T, HW, C, mode, groups, eps, reinterpret_cast<float2*>(stats), v4, s);
  return hipGetLastError();
}

template <int V, class TI>
static void run_norm_posconv(const void* x, int B, int T_in, int T_out, int H, int W, int C, int mode,
                             const float2* st, const float* scale, const float* bias, const float* pk,
                             const float* pb, void* out, hipStream_t s) {
  const long long total = (long long)B * T_in * H * W * (C / V);
  hipLaunchKernelGGL((block_norm_posconv_kernel<V, TI>), dim3(blocks_for(total, 256)), dim3(256), 0, s,
                     static_cast<const TI*>(x), T_in, T_out, H, W, C, mode, st, scale, bias, pk, pb,
                     static_cast<TI*>(out), total);
}

hipError_t launch_block_norm_posconv(const void* x, int dtype, int B, int T_in, int T_out, int H, int W, int C,
                                     int mode, const float* stats, const float* scale, const float* bias,
                                     const float* pk, const float* pb, void* out, hipStream_t s) {
  if ((long long)B * T_out * H * W * C == 0) return hipSuccess;
  const auto* st = reinterpret_cast<const float2*>(stats);
  const bool v4 = vec4_ok(dtype, C, {x, out}, {scale, bias, pk, pb});
  if (dtype == 0 && v4)
    run_norm_posconv<4, float>(x, B, T_in, T_out, H, W, C, mode, st, scale, bias, pk, pb, out, s);
  else if (dtype == 0)
    run_norm_posconv<1, float>(x, B, T_in, T_out, H, W, C, mode, st, scale, bias, pk, pb, out, s);
  else if (v4)
    run_norm_posconv<4, uint16_t>(x, B, T_in, T_out, H, W, C, mode, st, scale, bias, pk, pb, out, s);
  else
    run_norm_posconv<1, uint16_t>(x, B, T_in, T_out, H, W, C, mode, st, scale, bias, pk, pb, out, s);
  return hipGetLastError();
}

template <int V, class TI>
static void run_layer_norm(const void* x, long long M, int C, float eps, const float* scale, const float* bias,
                           int pre, int post, void* out, hipStream_t s) {
  const int nvec = (C + V - 1) / V;
  int L = 1;
  while (L < 64 && L * 2 < nvec) L *= 2;       // one to two vectors per lane while a wave holds the row
  const int nv = (nvec + L - 1) / L;
  const dim3 grid(blocks_for(M, 256 / L));
#define CSSM_LN_CASE(NV_)                                                                                           \
  hipLaunchKernelGGL((layer_norm_kernel<V, NV_, TI>), grid, dim3(256), 0, s, static_cast<const TI*>(x), M, C, L, eps, \
                     scale, bias, pre, post, static_cast<TI*>(out))
  if (nv <= 2)
    CSSM_LN_CASE(2);
  else if (nv <= 4)
    CSSM_LN_CASE(4);
  else
    CSSM_LN_CASE(8);
#undef CSSM_LN_CASE
}

// rows of up to 64 lanes x 8 vectors: 2048 channels in 4-element vectors, else 512
bool layer_norm_supported(int dtype, int C, const void* x, const float* scale, const float* bias, const void* out) {
  return C <= (vec4_ok(dtype, C, {x, out}, {scale, bias}) ? 2048 : 512);
}

hipError_t launch_layer_norm(const void* x, int dtype, long long M, int C, float eps, const float* scale,
                             const float* bias, int pre, int post, void* out, hipStream_t s) {
  if (M == 0) return hipSuccess;
  if (!layer_norm_supported(dtype, C, x, scale, bias, out)) return hipErrorInvalidValue;
  const bool v4 = vec4_ok(dtype, C, {x, out}, {scale, bias});
  if (dtype == 0 && v4)
    run_layer_norm<4, float>(x, M, C, eps, scale, bias, pre, post, out, s);
  else if (dtype == 0)
    run_layer_norm<1, float>(x, M, C, eps, scale, bias, pre, post, out, s);
  else if (v4)
    run_layer_norm<4, uint16_t>(x, M, C, eps, scale, bias, pre, post, out, s);
  else
    run_layer_norm<1, uint16_t>(x, M, C, eps, scale, bias, pre, post, out, s);
  return hipGetLastError();
}

bool mlp_dwconv_supported(long long N, int H, int W, int C) {
  return N > 0 && H > 0 && W > 0 && C > 0 && C % 32 == 0 && W <= 64 && H <= 4096 && C / 32 <= 65535 &&
         N * H <= 0x7fffffffLL;
}

hipError_t launch_mlp_dwconv(const float* x, int N, int H, int W, int C, const float* k3, const float* bias, float* out,
                             hipStream_t s) {
  if (!mlp_dwconv_supported(N, H, W, C)) return hipErrorInvalidValue;
  // R + 2 rows in kMlpPix pixels, all H where they fit (no halo rows then)
  const int fit = kMlpPix / W, R = H <= fit ? H : fit - 2, tiles = (H + R - 1) / R;
  hipLaunchKernelGGL(mlp_dwconv_kernel, dim3(unsigned((long long)N * tiles), unsigned(C / 32)), dim3(256),
                     size_t(R == H ? H : R + 2) * W * 128, s, x, H, W, C, R, tiles, k3, bias, out);
  return hipGetLastError();
}

hipError_t launch_block_residual(const void* res, int T_res, const void* y, int T_y, int dtype, int B, int T_out,
                                 int H, int W, int C, int act, void* out, hipStream_t s) {
  const int HWC = H * W * C;
  const long long total = (long long)B * T_out * HWC;
  if (total == 0) return hipSuccess;
  if (dtype == 0)
    hipLaunchKernelGGL(block_residual_kernel<float>, dim3(blocks_for(total, 256)), dim3(256), 0, s,
                       static_cast<const float*>(res), T_res, static_cast<const float*>(y), T_y, T_out, HWC, act,
                       static_cast<float*>(out), total);
  else
    hipLaunchKernelGGL(block_residual_kernel<uint16_t>, dim3(blocks_for(total, 256)), dim3(256), 0, s,
                       static_cast<const uint16_t*>(res), T_res, static_cast<const uint16_t*>(y), T_y, T_out, HWC,
                       act, static_cast<uint16_t*>(out), total);
  return hipGetLastError();
}

}  // namespace cssm
