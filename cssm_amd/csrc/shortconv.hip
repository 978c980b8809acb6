// Factored short convolution of GatedCSSM on plane-major x_main (gfx950):
//   s_t   = DWConv_{ks x ks, SAME}(x_t) + b_s          (cssm.py:487-492)
//   o_t   = sum_{j < kt} w_t[j] s_{t - kt + 1 + j} + b_t (zeros for t < 0; cssm.py:494-500)
//   u_t   = SiLU(o_t)                                   (cssm.py:502)
//   ctx_t = mean_{h,w} u_t                              (cssm.py:536)
// Either convolution may be absent (ks = 0 / kt = 0).  short_conv_planes runs the
// cell's own sizes (ks 0 or 3, kt <= 4, planes up to 128 x 128); short_conv_kernel,
// one block per (b, c) plane sequence with threads striding over pixels and every tap
// read from global memory, takes the rest.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "launch.h"

namespace cssm {

__device__ __forceinline__ float sc_ld(const float* p, size_t i) { return p[i]; }
__device__ __forceinline__ float sc_ld(const uint16_t* p, size_t i) { return __uint_as_float(uint32_t(p[i]) << 16); }
__device__ __forceinline__ void sc_st(float* p, size_t i, float v) { p[i] = v; }
__device__ __forceinline__ void sc_st(uint16_t* p, size_t i, float v) {
  uint32_t x = __float_as_uint(v);
  if ((x & 0x7f800000u) == 0x7f800000u) {
    p[i] = uint16_t((x >> 16) | ((x & 0x007fffffu) ? 0x40u : 0u));
  } else {
    x += 0x7fffu + ((x >> 16) & 1u);
    p[i] = uint16_t(x >> 16);
  }
}

template <class TI, class TO>
__global__ void __launch_bounds__(256)
short_conv_kernel(const TI* __restrict__ x, int T, int C, int H, int W, int ks, const float* __restrict__ ws,
                  const float* __restrict__ bs, int kt, const float* __restrict__ wt, const float* __restrict__ bt,
                  TO* __restrict__ u, float* __restrict__ ctx) {
  __shared__ float red[4];
  const int b = blockIdx.x / C, c = blockIdx.x % C;
  const int HW = H * W;
  const int lo = (ks - 1) / 2;
  const float bsc = (ks > 0) ? bs[c] : 0.0f;
  const float btc = (kt > 0) ? bt[c] : 0.0f;
  auto plane = [&](int t) -> size_t { return ((size_t(b) * T + t) * C + c) * size_t(HW); };
  // spatial stage at step t, pixel (h, w); HWIO kernel (ks, ks, 1, C)
  auto spatial = [&](int t, int h, int w) -> float {
    const size_t base = plane(t);
    if (ks == 0) return sc_ld(x, base + size_t(h) * W + w);
    float acc = bsc;
    for (int i = 0; i < ks; ++i) {
      const int hh = h + i - lo;
      if (hh < 0 || hh >= H) continue;
      for (int j = 0; j < ks; ++j) {
        const int ww = w + j - lo;
        if (ww < 0 || ww >= W) continue;
        acc = fmaf(sc_ld(x, base + size_t(hh) * W + ww), ws[(i * ks + j) * C + c], acc);
      }
    }
    return acc;
  };
  for (int t = 0; t < T; ++t) {
    float csum = 0.0f;
    for (int p = threadIdx.x; p < HW; p += blockDim.x) {
      const int h = p / W, w = p % W;
      float o;
      if (kt > 0) {
        o = btc;
        for (int j = 0; j < kt; ++j) {
          const int ts = t - kt + 1 + j;
          if (ts >= 0) o = fmaf(wt[j * C + c], spatial(ts, h, w), o);
        }
      } else {
        o = spatial(t, h, w);
      }
      const float v = o / (1.0f + expf(-o));
      sc_st(u, plane(t) + p, v);
      csum += v;
    }
    for (int off = 32; off > 0; off >>= 1) csum += __shfl_down(csum, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = csum;
    __syncthreads();
    if (threadIdx.x == 0 && ctx != nullptr) {
      float s = 0.0f;
      for (int i = 0; i < int(blockDim.x >> 6); ++i) s += red[i];
      ctx[(size_t(b) * T + t) * C + c] = s / float(HW);
    }
    __syncthreads();
  }
}

// Whole planes per workgroup, LP threads (a power of two) per plane with PX pixels each,
// walking a chunk of the frames in order.  A frame's plane goes through LDS with a zero
// border (NB buffers; the next frame's loads are in flight meanwhile), its 3 x 3 sums s_t are
// taken once and the last three frames' kept in registers for the temporal taps.  The
// one-pass-per-tap kernel above reads 9 kt values per output through L1 instead, and a
// block per plane leaves most CUs idle at small B C: frames are therefore dealt in chunks of
// tlen to gridDim.y (each starts kt - 1 frames early, spatial sums only).  Same sums in the
// same order as the kernel above, so the same results.  One read and one write of x: 1024
// frames x 256 planes of 16 x 16 in 216 us (2.5 TB/s; the kernel above 5.75 ms), 512 frames x
// 128 planes of 14 x 14 in 49 us (331 us), 512 x 32 of 32 x 32 in 57 us (436 us).
// pre != 0 stores o_t instead of u_t (ctx stays the mean of u_t).
template <int KS, int PX, int NT, int NB, int LDSF, class TI, class TO>
__global__ void __launch_bounds__(NT)
short_conv_planes(const TI* __restrict__ x, long long P, int T, int C, int H, int W, const float* __restrict__ ws,
                  const float* __restrict__ bs, int kt, const float* __restrict__ wt, const float* __restrict__ bt,
                  TO* __restrict__ u, float* __restrict__ ctx, int LP, int tlen, int pre, int still) {
  __shared__ float buf[KS ? NB * LDSF : 1];
  __shared__ float red[2][NT / 64];
  const int tid = threadIdx.x, NPL = NT / LP, pl = tid / LP, li = tid % LP;
  const int HW = H * W, RS = W + 2, PS = (H + 2) * RS;
  const long long plane = (long long)blockIdx.x * NPL + pl;
  const bool live = plane < P;
  const long long b = live ? plane / C : 0;
  const int c = live ? int(plane % C) : 0;
  const size_t base = (size_t(b) * T * C + c) * HW, tstep = size_t(C) * HW;
  const size_t xbase = still ? (size_t(b) * C + c) * HW : base, xstep = still ? 0 : tstep;   // one frame for all
  float k9[9], kt4[4], bsc = 0.0f, btc = 0.0f;
  if (KS) {
#pragma unroll
    for (int i = 0; i < 9; ++i) k9[i] = ws[i * C + c];
    bsc = bs[c];
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) kt4[j] = j < kt ? wt[(kt - 1 - j) * C + c] : 0.0f;   // by lag
  if (kt > 0) btc = bt[c];
  int off[PX];     // LDS slot of the pixel's upper left neighbour
#pragma unroll
  for (int k = 0; k < PX; ++k) {
    const int p = li + k * LP;
    off[k] = pl * PS + (p / W) * RS + p % W;
  }
  if (KS) {
    for (int i = tid; i < NB * LDSF; i += NT) buf[i] = 0.0f;
    __syncthreads();
  }
  const int t0 = int(blockIdx.y) * tlen, t1 = t0 + tlen < T ? t0 + tlen : T;
  const int ts = kt > 1 ? (t0 - (kt - 1) > 0 ? t0 - (kt - 1) : 0) : t0;
  float nx[PX], h1[PX], h2[PX], h3[PX];
  auto load = [&](int t) {
#pragma unroll
    for (int k = 0; k < PX; ++k) {
      const int p = li + k * LP;
      nx[k] = live && p < HW ? sc_ld(x, xbase + size_t(t) * xstep + p) : 0.0f;
    }
  };
#pragma unroll
  for (int k = 0; k < PX; ++k) h1[k] = h2[k] = h3[k] = 0.0f;
  load(ts);
  // the mean of frame t from the waves' sums (LP > 64), one barrier after they were written
  auto finish_ctx = [&](int t) {
    if (ctx != nullptr && LP > 64 && li == 0 && live) {
      float sum = 0.0f;
      for (int i = 0; i < LP / 64; ++i) sum += red[t & 1][tid / 64 + i];
      ctx[(size_t(b) * T + t) * C + c] = sum / float(HW);
    }
  };
  for (int t = ts; t < t1; ++t) {
    float* bt_ = buf + (NB == 2 ? (t & 1) * LDSF : 0);
    float s[PX];
    if (KS) {
#pragma unroll
      for (int k = 0; k < PX; ++k)
        if (li + k * LP < HW) bt_[off[k] + RS + 1] = nx[k];
    } else {
#pragma unroll
      for (int k = 0; k < PX; ++k) s[k] = nx[k];
    }
    if (KS || LP > 64) __syncthreads();
    if (t > t0) finish_ctx(t - 1);
    if (t + 1 < t1) load(t + 1);
    if (KS) {
#pragma unroll
      for (int k = 0; k < PX; ++k) {
        float acc = bsc;
        const float* q = bt_ + (li + k * LP < HW ? off[k] : 0);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int j = 0; j < 3; ++j) acc = fmaf(q[i * RS + j], k9[i * 3 + j], acc);
        s[k] = acc;
      }
    }
    if (t >= t0) {
      float csum = 0.0f;
      TO* ut = u + base + size_t(t) * tstep;
#pragma unroll
      for (int k = 0; k < PX; ++k) {
        const int p = li + k * LP;
        float o = s[k];
        if (kt > 0) {   // oldest frame first; frames before the first are left out
          o = btc;
          if (kt > 3 && t >= 3) o = fmaf(kt4[3], h3[k], o);
          if (kt > 2 && t >= 2) o = fmaf(kt4[2], h2[k], o);
          if (kt > 1 && t >= 1) o = fmaf(kt4[1], h1[k], o);
          o = fmaf(kt4[0], s[k], o);
        }
        const float v = o / (1.0f + expf(-o));
        if (live && p < HW) {
          sc_st(ut, size_t(p), pre ? o : v);
          csum += v;
        }
      }
      if (ctx != nullptr) {
        for (int o = (LP < 64 ? LP : 64) / 2; o > 0; o >>= 1) csum += __shfl_xor(csum, o, 64);
        if (LP <= 64) {
          if (li == 0 && live) ctx[(size_t(b) * T + t) * C + c] = csum / float(HW);
        } else if ((tid & 63) == 0) {
          red[t & 1][tid / 64] = csum;
        }
      }
    }
#pragma unroll
    for (int k = 0; k < PX; ++k) {
      h3[k] = h2[k];
      h2[k] = h1[k];
      h1[k] = s[k];
    }
    if (KS && NB == 1) __syncthreads();   // one buffer: its readers are done
  }
  if (LP > 64) {
    __syncthreads();
    finish_ctx(t1 - 1);
  }
}

// LDS floats of a plane with its border, per kernel class
constexpr int kScSmall = 4096, kScMid = 4400, kScLarge = 16900;

// the kernel class of a call (0: 256 threads, 4 pixels each; 1: 1024, 4; 2: 1024, 16), threads per plane and
// frames per workgroup: all of them when the planes alone give every CU its waves (16 per CU), else
// chunks of at least 8 (a chunk reads kt - 1 frames more)
struct ScShape {
  int cls, LP, tlen;
};
static ScShape sc_shape(int B, int T, int C, int H, int W) {
  const long long HW = (long long)H * W, ps = (long long)(H + 2) * (W + 2);
  ScShape r{0, 1, T};
  while (r.LP < 256 && r.LP * 4 < HW) r.LP *= 2;
  if (!(HW <= 1024 && (256 / r.LP) * ps <= kScSmall)) {
    r.cls = HW <= 4096 && ps <= kScMid ? 1 : 2;
    r.LP = 1024;
  }
  const int NT = r.cls == 0 ? 256 : 1024;
  const long long P = (long long)B * C, groups = (P + NT / r.LP - 1) / (NT / r.LP);
  const long long want = 256LL * 1024 / NT;
  long long chunks = groups >= want ? 1 : (want + groups - 1) / groups;
  if (chunks > (T + 7) / 8) chunks = (T + 7) / 8;
  r.tlen = int((T + chunks - 1) / chunks);
  return r;
}

template <int PX, int NT, int NB, int LDSF, class TI, class TO>
static void run_short_conv_planes(const TI* x, int B, int T, int C, int H, int W, int ks, const float* ws,
                                  const float* bs, int kt, const float* wt, const float* bt, TO* u, float* ctx,
                                  const ScShape& r, int pre, int still, hipStream_t s) {
  const long long P = (long long)B * C;
  const dim3 grid(unsigned((P + NT / r.LP - 1) / (NT / r.LP)), unsigned((T + r.tlen - 1) / r.tlen));
  if (ks == 3)
    hipLaunchKernelGGL((short_conv_planes<3, PX, NT, NB, LDSF, TI, TO>), grid, dim3(NT), 0, s, x, P, T, C, H, W, ws,
                       bs, kt, wt, bt, u, ctx, r.LP, r.tlen, pre, still);
  else
    hipLaunchKernelGGL((short_conv_planes<0, PX, NT, NB, LDSF, TI, TO>), grid, dim3(NT), 0, s, x, P, T, C, H, W, ws,
                       bs, kt, wt, bt, u, ctx, r.LP, r.tlen, pre, still);
}

template <class TI, class TO>
static void run_short_conv(const TI* x, int B, int T, int C, int H, int W, int ks, const float* ws, const float* bs,
                           int kt, const float* wt, const float* bt, TO* u, float* ctx, int pre, int still, hipStream_t s) {
  const ScShape r = sc_shape(B, T, C, H, W);
  if (r.cls == 0)
    run_short_conv_planes<4, 256, 2, kScSmall>(x, B, T, C, H, W, ks, ws, bs, kt, wt, bt, u, ctx, r, pre, still, s);
  else if (r.cls == 1)
    run_short_conv_planes<4, 1024, 2, kScMid>(x, B, T, C, H, W, ks, ws, bs, kt, wt, bt, u, ctx, r, pre, still, s);
  else
    run_short_conv_planes<16, 1024, 1, kScLarge>(x, B, T, C, H, W, ks, ws, bs, kt, wt, bt, u, ctx, r, pre, still, s);
}

// where short_conv_planes applies (else the general kernel, which has no pre form)
bool short_conv_planes_supported(int T, int H, int W, int ks, int kt) {
  return (ks == 0 || ks == 3) && kt <= 4 && (long long)H * W <= 16384 && (long long)(H + 2) * (W + 2) <= kScLarge &&
         T <= 65535 * 8;
}

// Adjoint of short_conv_planes' convolutions: from do = dL/d(pre-activation) of every frame,
//   ds_t = sum_l w_l do_{t+l} (w_l the tap of lag l),  dx_t = the 3 x 3 conv of ds_t with flipped taps,
//   dw_l = sum s_t do_{t+l},  db_t = sum do,  dW[i][j] = sum ds x shifted,  db_s = sum ds
// and the sum of dx (the projection's bias gradient).  The same plane groups and frame chunks, walked
// backwards with do of the next three frames in registers (a chunk starts kt - 1 frames late); x_t and
// ds_t go through LDS with zero borders, s_t is taken from x_t again.  Each plane's sixteen sums leave
// once per chunk: sums (chunks, B C, 16) = [W 9, b_s, w_0..w_3 by lag, b_t, dx].  Reads x and do, writes
// dx once: 256 frames x 64 planes of 32 x 32 in 72 us (2.8 TB/s; the library's depthwise conv, its im2col
// weight gradient and the elementwise passes around them 4.5 ms).
template <int KS, int PX, int NT, int LDSF>
__global__ void __launch_bounds__(NT)
short_conv_planes_bwd(const float* __restrict__ x, const float* __restrict__ dout, long long P, int T, int C, int H,
                      int W, const float* __restrict__ ws, const float* __restrict__ bs, int kt,
                      const float* __restrict__ wt, float* __restrict__ dx, long long dx_fs, float* __restrict__ sums,
                      int LP, int tlen) {
  __shared__ float bx[KS ? LDSF : 1], bd[KS ? LDSF : 1];
  __shared__ float red[16][NT / 64];
  const int tid = threadIdx.x, NPL = NT / LP, pl = tid / LP, li = tid % LP;
  const int HW = H * W, RS = W + 2, PS = (H + 2) * RS;
  const long long plane = (long long)blockIdx.x * NPL + pl;
  const bool live = plane < P;
  const long long b = live ? plane / C : 0;
  const int c = live ? int(plane % C) : 0;
  const size_t base = (size_t(b) * T * C + c) * HW, tstep = size_t(C) * HW;
  float* dxp = dx + size_t(b) * T * dx_fs + size_t(c) * HW;
  float k9[9], kt4[4], bsc = 0.0f;
  if (KS) {
#pragma unroll
    for (int i = 0; i < 9; ++i) k9[i] = ws[i * C + c];
    bsc = bs[c];
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) kt4[j] = j < kt ? wt[(kt - 1 - j) * C + c] : 0.0f;
  int off[PX];
#pragma unroll
  for (int k = 0; k < PX; ++k) {
    const int p = li + k * LP;
    off[k] = pl * PS + (p < HW ? (p / W) * RS + p % W : 0);
  }
  if (KS) {
    for (int i = tid; i < LDSF; i += NT) bx[i] = bd[i] = 0.0f;
    __syncthreads();
  }
  const int t0 = int(blockIdx.y) * tlen, t1 = t0 + tlen < T ? t0 + tlen : T;
  int te = t1 - 1 + (kt > 1 ? kt - 1 : 0);
  if (te > T - 1) te = T - 1;
  float acc[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) acc[j] = 0.0f;
  float d1[PX], d2[PX], d3[PX], nd[PX], nx[PX];   // do of frames t + 1, t + 2, t + 3; the next frame's loads
#pragma unroll
  for (int k = 0; k < PX; ++k) d1[k] = d2[k] = d3[k] = 0.0f;
  auto load = [&](int t) {
#pragma unroll
    for (int k = 0; k < PX; ++k) {
      const int p = li + k * LP;
      const bool ok = live && p < HW;
      nd[k] = ok ? dout[base + size_t(t) * tstep + p] : 0.0f;
      nx[k] = ok && t < t1 ? x[base + size_t(t) * tstep + p] : 0.0f;
    }
  };
  load(te);
  for (int t = te; t >= t0; --t) {
    float d0[PX], ds[PX], xv[PX];
#pragma unroll
    for (int k = 0; k < PX; ++k) {
      d0[k] = nd[k];
      xv[k] = nx[k];
    }
    if (t > t0) load(t - 1);
    if (t < t1) {
#pragma unroll
      for (int k = 0; k < PX; ++k) {
        ds[k] = d0[k];
        if (kt > 0) {
          ds[k] = kt4[0] * d0[k];
          if (kt > 1) ds[k] = fmaf(kt4[1], d1[k], ds[k]);
          if (kt > 2) ds[k] = fmaf(kt4[2], d2[k], ds[k]);
          if (kt > 3) ds[k] = fmaf(kt4[3], d3[k], ds[k]);
        }
        if (KS && li + k * LP < HW) {
          bx[off[k] + RS + 1] = xv[k];
          bd[off[k] + RS + 1] = ds[k];
        }
      }
      if (KS) __syncthreads();
      float* dt = dxp + size_t(t) * dx_fs;
#pragma unroll
      for (int k = 0; k < PX; ++k) {
        const int p = li + k * LP;
        float s = xv[k], g = ds[k];
        if (KS) {
          s = bsc;
          g = 0.0f;
          const float* qx = bx + off[k];
          const float* qd = bd + off[k];
#pragma unroll
          for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) {
              const float v = qx[i * RS + j];
              s = fmaf(v, k9[i * 3 + j], s);
              acc[i * 3 + j] = fmaf(ds[k], v, acc[i * 3 + j]);
              g = fmaf(qd[(2 - i) * RS + 2 - j], k9[i * 3 + j], g);
            }
          acc[9] += ds[k];
        }
        if (!(live && p < HW)) s = g = 0.0f;
        acc[10] = fmaf(s, d0[k], acc[10]);
        acc[11] = fmaf(s, d1[k], acc[11]);
        acc[12] = fmaf(s, d2[k], acc[12]);
        acc[13] = fmaf(s, d3[k], acc[13]);
        acc[14] += d0[k];
        acc[15] += g;
        if (live && p < HW) dt[p] = g;
      }
      if (KS) __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < PX; ++k) {
      d3[k] = d2[k];
      d2[k] = d1[k];
      d1[k] = d0[k];
    }
  }
#pragma unroll
  for (int j = 0; j < 16; ++j)
    for (int o = (LP < 64 ? LP : 64) / 2; o > 0; o >>= 1) acc[j] += __shfl_xor(acc[j], o, 64);
  float* out = sums + (size_t(blockIdx.y) * P + (live ? plane : 0)) * 16;
  if (LP <= 64) {
    if (li == 0 && live)
#pragma unroll
      for (int j = 0; j < 16; ++j) out[j] = acc[j];
    return;
  }
  if ((tid & 63) == 0)
#pragma unroll
    for (int j = 0; j < 16; ++j) red[j][tid / 64] = acc[j];
  __syncthreads();
  if (live && li < 16) {
    float v = 0.0f;
    for (int i = 0; i < LP / 64; ++i) v += red[li][pl * (LP / 64) + i];
    out[li] = v;
  }
}

int short_conv_bwd_chunks(int B, int T, int C, int H, int W) {
  const ScShape r = sc_shape(B, T, C, H, W);
  return (T + r.tlen - 1) / r.tlen;
}

template <int KS, int PX, int NT, int LDSF>
static void run_short_conv_bwd(const float* x, const float* dout, int B, int T, int C, int H, int W, const float* ws,
                               const float* bs, int kt, const float* wt, float* dx, long long dx_fs, float* sums,
                               const ScShape& r, hipStream_t s) {
  const long long P = (long long)B * C;
  const dim3 grid(unsigned((P + NT / r.LP - 1) / (NT / r.LP)), unsigned((T + r.tlen - 1) / r.tlen));
  hipLaunchKernelGGL((short_conv_planes_bwd<KS, PX, NT, LDSF>), grid, dim3(NT), 0, s, x, dout, P, T, C, H, W, ws, bs,
                     kt, wt, dx, dx_fs, sums, r.LP, r.tlen);
}

hipError_t launch_short_conv_bwd(const float* x, const float* dout, int B, int T, int C, int H, int W, int ks,
                                 const float* ws, const float* bs, int kt, const float* wt, float* dx,
                                 long long dx_fs, float* sums, hipStream_t s) {
  if (!short_conv_planes_supported(T, H, W, ks, kt)) return hipErrorInvalidValue;
  const ScShape r = sc_shape(B, T, C, H, W);
#define CSSM_SCB(KS_)                                                                                                \
  if (r.cls == 0) run_short_conv_bwd<KS_, 4, 256, kScSmall>(x, dout, B, T, C, H, W, ws, bs, kt, wt, dx, dx_fs, sums, r, s); \
  else if (r.cls == 1) run_short_conv_bwd<KS_, 4, 1024, kScMid>(x, dout, B, T, C, H, W, ws, bs, kt, wt, dx, dx_fs, sums, r, s); \
  else run_short_conv_bwd<KS_, 16, 1024, kScLarge>(x, dout, B, T, C, H, W, ws, bs, kt, wt, dx, dx_fs, sums, r, s);
  if (ks == 3) {
    CSSM_SCB(3)
  } else {
    CSSM_SCB(0)
  }
#undef CSSM_SCB
  return hipGetLastError();
}

hipError_t launch_short_conv(const void* x, int in_dtype, int B, int T, int C, int H, int W, int ks, const float* ws,
                             const float* bs, int kt, const float* wt, const float* bt, void* u, int out_dtype,
                             float* ctx, int pre, hipStream_t s, bool still) {
  if (short_conv_planes_supported(T, H, W, ks, kt)) {
    if (in_dtype == 0 && out_dtype == 0)
      run_short_conv(static_cast<const float*>(x), B, T, C, H, W, ks, ws, bs, kt, wt, bt, static_cast<float*>(u), ctx,
                     pre, still, s);
    else if (in_dtype == 0)
      run_short_conv(static_cast<const float*>(x), B, T, C, H, W, ks, ws, bs, kt, wt, bt, static_cast<uint16_t*>(u),
                     ctx, pre, still, s);
    else if (out_dtype == 0)
      run_short_conv(static_cast<const uint16_t*>(x), B, T, C, H, W, ks, ws, bs, kt, wt, bt, static_cast<float*>(u),
                     ctx, pre, still, s);
    else
      run_short_conv(static_cast<const uint16_t*>(x), B, T, C, H, W, ks, ws, bs, kt, wt, bt,
                     static_cast<uint16_t*>(u), ctx, pre, still, s);
    return hipGetLastError();
  }
  if (pre || still) return hipErrorInvalidValue;
  const dim3 grid(unsigned(B * C)), block(256);
  if (in_dtype == 0 && out_dtype == 0)
    hipLaunchKernelGGL((short_conv_kernel<float, float>), grid, block, 0, s, static_cast<const float*>(x), T, C, H, W,
                       ks, ws, bs, kt, wt, bt, static_cast<float*>(u), ctx);
  else if (in_dtype == 0)
    hipLaunchKernelGGL((short_conv_kernel<float, uint16_t>), grid, block, 0, s, static_cast<const float*>(x), T, C, H,
                       W, ks, ws, bs, kt, wt, bt, static_cast<uint16_t*>(u), ctx);
  else if (out_dtype == 0)
    hipLaunchKernelGGL((short_conv_kernel<uint16_t, float>), grid, block, 0, s, static_cast<const uint16_t*>(x), T, C,
                       H, W, ks, ws, bs, kt, wt, bt, static_cast<float*>(u), ctx);
  else
    hipLaunchKernelGGL((short_conv_kernel<uint16_t, uint16_t>), grid, block, 0, s, static_cast<const uint16_t*>(x), T,
                       C, H, W, ks, ws, bs, kt, wt, bt, static_cast<uint16_t*>(u), ctx);
  return hipGetLastError();
}

}  // namespace cssm
