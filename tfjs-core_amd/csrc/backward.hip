// Memory-bound backward kernels of the NHWC image ops: depthwiseConv2DDerInput /
// depthwiseConv2DDerFilter (backend_cpu.ts:2037-2150 of the reference) and maxPoolBackprop /
// avgPoolBackprop (:2347-2509).  (conv2dDerInput / conv2dDerFilter are products and live
// with the dense kernels.)
//
// The gradients with respect to an image are gathers: one lane per dx element, output
// channel fastest, so a wavefront reads runs of consecutive dy elements.  The gradient with
// respect to the depthwise filter is a reduction over every output pixel: lanes run along
// the channels, workgroups split the pixels, and a second kernel adds the partial sums in a
// fixed order, so the result does not depend on scheduling.
#include <algorithm>
#include <cstring>

#include "tfhip_internal.h"

namespace tfhip {

// dx[n, xr, xc, d1] = sum over the output pixels (yr, yc) whose window covers (xr, xc), and
// over the channel multiplier, of dy * w; taps in the order of the reference's loops (output
// row, output column, multiplier).  Accumulated in double, stored once, like the reference.
__global__ void depthwise_der_input_kernel(const float* dy, const float* w, float* dx,
                                           const tfhip_conv2d_info ci, int ch_mul) {
  const int64_t total = (int64_t)ci.batch * ci.in_h * ci.in_w * ci.in_c;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int top_pad = ci.filter_h - 1 - ci.pad_top, left_pad = ci.filter_w - 1 - ci.pad_left;
  for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += stride) {
    const int d1 = (int)(g % ci.in_c);
    int64_t t = g / ci.in_c;
    const int xc = (int)(t % ci.in_w);
    t /= ci.in_w;
    const int xr = (int)(t % ci.in_h);
    const int n = (int)(t / ci.in_h);
    const int xr_corner = xr - top_pad, xc_corner = xc - left_pad;
    double dot = 0.0;
    for (int wr = 0; wr < ci.filter_h; wr++) {
      const int num_r = xr_corner + wr;  // = yr * stride_h
      if (num_r < 0 || num_r % ci.stride_h != 0) continue;
      const int yr = num_r / ci.stride_h;
      if (yr >= ci.out_h) continue;
      for (int wc = 0; wc < ci.filter_w; wc++) {
        const int num_c = xc_corner + wc;
        if (num_c < 0 || num_c % ci.stride_w != 0) continue;
        const int yc = num_c / ci.stride_w;
        if (yc >= ci.out_w) continue;
        const float* dyp =
            dy + (((int64_t)n * ci.out_h + yr) * ci.out_w + yc) * ci.out_c + (int64_t)d1 * ch_mul;
        const float* wp = w + (((int64_t)(ci.filter_h - 1 - wr) * ci.filter_w +
                                (ci.filter_w - 1 - wc)) * ci.in_c + d1) * ch_mul;
        for (int dm = 0; dm < ch_mul; dm++) dot += (double)dyp[dm] * (double)wp[dm];
      }
    }
    dx[g] = (float)dot;
  }
}

// Partial sums of dW over a slice of the output pixels.  grid = (channel blocks of 64,
// filter taps, pixel slices); a workgroup's 4 wavefronts take every 4th pixel of the slice,
// lane = output channel d2 (so dy, and for multiplier 1 also x, are read in 256-byte runs).
// partial[slice][tap][d2] in double.
__global__ __launch_bounds__(256) void depthwise_der_filter_partial_kernel(
    const float* x, const float* dy, double* partial, const tfhip_conv2d_info ci, int ch_mul,
    int64_t pixels_per_slice) {
  __shared__ double red[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int d2 = blockIdx.x * 64 + lane;
  const int tap = blockIdx.y, wr = tap / ci.filter_w, wc = tap % ci.filter_w;
  const int64_t pixels = (int64_t)ci.batch * ci.out_h * ci.out_w;
  const int64_t p0 = (int64_t)blockIdx.z * pixels_per_slice;
  const int64_t p1 = p0 + pixels_per_slice < pixels ? p0 + pixels_per_slice : pixels;
  const bool live = d2 < ci.out_c;
  const int d1 = live ? d2 / ch_mul : 0;
  double dot = 0.0;
  for (int64_t px = p0 + wave; px < p1; px += 4) {
    const int yc = (int)(px % ci.out_w);
    const int64_t t = px / ci.out_w;
    const int yr = (int)(t % ci.out_h);
    const int n = (int)(t / ci.out_h);
    const int xr = wr + yr * ci.stride_h - ci.pad_top, xc = wc + yc * ci.stride_w - ci.pad_left;
    if ((unsigned)xr >= (unsigned)ci.in_h || (unsigned)xc >= (unsigned)ci.in_w || !live) continue;
    dot += (double)x[(((int64_t)n * ci.in_h + xr) * ci.in_w + xc) * ci.in_c + d1] *
           (double)dy[px * ci.out_c + d2];
  }
  red[wave][lane] = dot;
  __syncthreads();
  if (wave == 0 && live)
    partial[((int64_t)blockIdx.z * gridDim.y + tap) * ci.out_c + d2] =
        ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
}

// dW[tap][d1][dm] = sum of the slices' partial sums: a workgroup takes 32 elements, its 32 rows of
// lanes every 32nd slice with 8 loads in flight, and the 32 sums are added in ascending order.  One
// lane per element walking its slices alone was a chain of loads: 1152 elements of 512 slices took
// 94 us, 4 here; 896 slices take 5.8.
__global__ __launch_bounds__(1024) void depthwise_der_filter_finish_kernel(const double* partial, float* dw,
                                                                           int64_t w_n, int slices) {
  constexpr int ROWS = 32, UNROLL = 8;
  __shared__ double sums[ROWS][32];
  const int lane = threadIdx.x & 31, row = threadIdx.x >> 5;
  const int64_t g = (int64_t)blockIdx.x * 32 + lane;
  double s = 0.0;
  if (g < w_n)
    for (int i = row; i < slices; i += ROWS * UNROLL) {
      double v[UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; u++) v[u] = partial[(int64_t)min(i + u * ROWS, slices - 1) * w_n + g];
#pragma unroll
      for (int u = 0; u < UNROLL; u++) s += i + u * ROWS < slices ? v[u] : 0.0;
    }
  sums[row][lane] = s;
  __syncthreads();
  if (row == 0 && g < w_n) {
    for (int r = 1; r < ROWS; r++) s += sums[r][lane];
    dw[g] = (float)s;
  }
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Fast variants for channel multiplier 1, C % 4 == 0 and 16-byte aligned buffers: a lane owns
// 4 consecutive channels (16-byte accesses) and sums in float in the same tap order.
// S = 1, 2: the forward stride, known at compile time (no integer division); S = 0: any.
template <int S>
__global__ __launch_bounds__(256) void depthwise_der_input_vec_kernel(
    const float* __restrict__ dy, const float* __restrict__ w, float* __restrict__ dx,
    const tfhip_conv2d_info ci, uint32_t total, Divisor by_c4, Divisor by_w, Divisor by_h) {
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= total) return;
  uint32_t t = g;
  const int cq = (int)by_c4.divmod(t), xc = (int)by_w.divmod(t), xr = (int)by_h.divmod(t), n = (int)t;
  const int sh = S ? S : ci.stride_h, sw = S ? S : ci.stride_w;
  const int xr_corner = xr - (ci.filter_h - 1 - ci.pad_top);
  const int xc_corner = xc - (ci.filter_w - 1 - ci.pad_left);
  const float* dyn = dy + (int64_t)n * ci.out_h * ci.out_w * ci.out_c + cq * 4;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int wr = 0; wr < ci.filter_h; wr++) {
    const int num_r = xr_corner + wr;
    const int yr = num_r / sh;
    if (num_r < 0 || yr * sh != num_r || yr >= ci.out_h) continue;
    for (int wc = 0; wc < ci.filter_w; wc++) {
      const int num_c = xc_corner + wc;
      const int yc = num_c / sw;
      if (num_c < 0 || yc * sw != num_c || yc >= ci.out_w) continue;
      const f32x4 d = *reinterpret_cast<const f32x4*>(dyn + ((int64_t)yr * ci.out_w + yc) * ci.out_c);
      const f32x4 f = *reinterpret_cast<const f32x4*>(
          w + ((int64_t)(ci.filter_h - 1 - wr) * ci.filter_w + (ci.filter_w - 1 - wc)) * ci.in_c + cq * 4);
      acc += d * f;
    }
  }
  *reinterpret_cast<f32x4*>(dx + (int64_t)g * 4) = acc;
}

// dW of a 3x3 depthwise filter (multiplier 1) at stride S.  A lane owns a channel quad and walks the
// output rows of a column segment (a unit) with the nine taps' sums in registers: the window's rows
// stay in registers from one output pixel to the next, so a pixel costs 3 S loads of x and one of dy
// (those of the next row are in flight while a row is added), and neighbouring lanes share them in
// L1.  Rows and columns beyond the image read 0 through the buffer descriptor.  The lanes of
// a workgroup that share a quad are then added in a fixed order through LDS.
// partial[slice][tap][c] in double.  Bound by the one read of x and dy from memory:
// [32,56,56,128] 21.4 us (4.8 TB/s), at stride 2 13.8; ten loads a pixel, as below, 32.0 and 15.4.
template <int S>
__global__ __launch_bounds__(256) void depthwise3x3_der_filter_rows_kernel(
    const float* __restrict__ x, const float* __restrict__ dy, double* __restrict__ partial,
    const tfhip_conv2d_info ci, unsigned x_bytes, unsigned y_bytes, int quads_per_wave, int rows, uint32_t units,
    Divisor by_w, Divisor by_segs) {
  extern __shared__ __attribute__((aligned(16))) float red[];  // [256 lanes][9 taps][4]
  constexpr int NB = S + 3;             // row buffers: three in use, S on their way
  constexpr unsigned OOB = 0x80000000u;  // beyond any extent below 2 GiB
  const int tid = threadIdx.x;
  const int q_local = tid & (quads_per_wave - 1);       // quad within the channel block (a power of two)
  const int subs = 256 / quads_per_wave, sub = tid / quads_per_wave;
  const int c = (blockIdx.x * quads_per_wave + q_local) * 4;
  const __amdgpu_buffer_rsrc_t rx =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x), (short)0, (int)x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t ry =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(dy), (short)0, (int)y_bytes, 0x00020000);
  const unsigned x_row = (unsigned)ci.in_w * ci.in_c * 4u, y_row = (unsigned)ci.out_w * ci.out_c * 4u;
  f32x4 acc[9];
#pragma unroll
  for (int k = 0; k < 9; k++) acc[k] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (c < ci.in_c)
    for (uint32_t unit = blockIdx.y * subs + sub; unit < units; unit += gridDim.y * subs) {
      uint32_t t = unit;
      const int yc = (int)by_w.divmod(t), seg = (int)by_segs.divmod(t), n = (int)t;
      const int y0 = seg * rows, y1 = min(y0 + rows, ci.out_h);
      unsigned col[3];
#pragma unroll
      for (int j = 0; j < 3; j++) {
        const int xc = yc * S - ci.pad_left + j;
        col[j] = (unsigned)xc < (unsigned)ci.in_w ? ((unsigned)(n * ci.in_h * ci.in_w + xc) * ci.in_c + c) * 4u : OOB;
      }
      const unsigned y_at = ((unsigned)(n * ci.out_h * ci.out_w + yc) * ci.out_c + c) * 4u;
      f32x4 v[NB][3], d[NB];
      auto load_row = [&](int r, f32x4 (&to)[3]) {
        const bool ok = (unsigned)r < (unsigned)ci.in_h && r <= (y1 - 1) * S - ci.pad_top + 2;
#pragma unroll
        for (int j = 0; j < 3; j++)
          to[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                rx, (int)(ok && col[j] != OOB ? (unsigned)r * x_row + col[j] : OOB), 0, 0));
      };
      auto load_dy = [&](int y) {
        return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                             ry, (int)(y < y1 ? (unsigned)y * y_row + y_at : OOB), 0, 0));
      };
      const int first = y0 * S - ci.pad_top;
#pragma unroll
      for (int k = 0; k < 3; k++) load_row(first + k, v[k]);
      d[0] = load_dy(y0);
      for (int y = y0; y < y1; y += NB) {
#pragma unroll
        for (int u = 0; u < NB; u++) {
          if (y + u < y1) {
            const int r = (y + u) * S - ci.pad_top;
#pragma unroll
            for (int k = 0; k < S; k++) load_row(r + 3 + k, v[(u * S + 3 + k) % NB]);
            d[(u + 1) % NB] = load_dy(y + u + 1);
            __builtin_amdgcn_sched_barrier(0);  // loads first
#pragma unroll
            for (int i = 0; i < 3; i++)
#pragma unroll
              for (int j = 0; j < 3; j++) acc[i * 3 + j] += v[(u * S + i) % NB][j] * d[u];
          }
        }
      }
    }
#pragma unroll
  for (int k = 0; k < 9; k++) *reinterpret_cast<f32x4*>(red + (tid * 9 + k) * 4) = acc[k];
  __syncthreads();
  // thread -> (tap, quad): add the `subs` lanes of that quad in ascending order, in double
  for (int item = tid; item < 9 * quads_per_wave; item += 256) {
    const int k = item / quads_per_wave, q = item & (quads_per_wave - 1);
    const int oc = (blockIdx.x * quads_per_wave + q) * 4;
    if (oc >= ci.in_c) continue;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    for (int r = 0; r < subs; r++) {
      const float* p = red + ((r * quads_per_wave + q) * 9 + k) * 4;
      s0 += (double)p[0];
      s1 += (double)p[1];
      s2 += (double)p[2];
      s3 += (double)p[3];
    }
    double* out = partial + ((int64_t)blockIdx.y * 9 + k) * ci.in_c + oc;
    out[0] = s0;
    out[1] = s1;
    out[2] = s2;
    out[3] = s3;
  }
}

// The same at any other stride, and for operands of 2 GiB and more: a pass over the output pixels of a slice;
// a lane owns a channel quad and keeps the nine taps' sums, so dy is read once and the nine
// x vectors of a pixel come from neighbouring rows that stay in cache.  The lanes of a
// workgroup that share a quad (several pixels per wavefront when C / 4 < 64, and the four
// wavefronts) are then added in a fixed order through LDS.  partial[slice][tap][c] in double.
__global__ __launch_bounds__(256) void depthwise3x3_der_filter_partial_kernel(
    const float* __restrict__ x, const float* __restrict__ dy, double* __restrict__ partial,
    const tfhip_conv2d_info ci, int quads_per_wave, int64_t pixels_per_slice, Divisor by_w, Divisor by_h) {
  extern __shared__ __attribute__((aligned(16))) float red[];  // [256 lanes][9 taps][4]
  const int tid = threadIdx.x;
  const int c4 = ci.in_c / 4;
  const int q_local = tid % quads_per_wave;            // quad within the channel block
  const int sub = tid / quads_per_wave;                // which of the workgroup's pixel lanes
  const int subs = 256 / quads_per_wave;
  const int cq = blockIdx.x * quads_per_wave + q_local;
  const bool live = cq < c4;
  const int64_t pixels = (int64_t)ci.batch * ci.out_h * ci.out_w;
  const int64_t p0 = (int64_t)blockIdx.y * pixels_per_slice;
  const int64_t p1 = p0 + pixels_per_slice < pixels ? p0 + pixels_per_slice : pixels;
  f32x4 acc[9];
#pragma unroll
  for (int k = 0; k < 9; k++) acc[k] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (live) {
    for (int64_t px = p0 + sub; px < p1; px += subs) {
      uint32_t t = (uint32_t)px;
      const int yc = (int)by_w.divmod(t), yr = (int)by_h.divmod(t), n = (int)t;
      const f32x4 d = *reinterpret_cast<const f32x4*>(dy + px * ci.out_c + cq * 4);
      const int xr0 = yr * ci.stride_h - ci.pad_top, xc0 = yc * ci.stride_w - ci.pad_left;
      const float* xn = x + (int64_t)n * ci.in_h * ci.in_w * ci.in_c + cq * 4;
#pragma unroll
      for (int wr = 0; wr < 3; wr++) {
        const int xr = xr0 + wr;
#pragma unroll
        for (int wc = 0; wc < 3; wc++) {
          const int xc = xc0 + wc;
          f32x4 v = {0.f, 0.f, 0.f, 0.f};
          if ((unsigned)xr < (unsigned)ci.in_h && (unsigned)xc < (unsigned)ci.in_w)
            v = *reinterpret_cast<const f32x4*>(xn + ((int64_t)xr * ci.in_w + xc) * ci.in_c);
          acc[wr * 3 + wc] += v * d;
        }
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 9; k++) *reinterpret_cast<f32x4*>(red + (tid * 9 + k) * 4) = acc[k];
  __syncthreads();
  // thread -> (tap, quad): add the `subs` lanes of that quad in ascending order, in double
  for (int item = tid; item < 9 * quads_per_wave; item += 256) {
    const int k = item / quads_per_wave, q = item % quads_per_wave;
    const int c = (blockIdx.x * quads_per_wave + q) * 4;
    if (c >= ci.in_c) continue;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    for (int r = 0; r < subs; r++) {
      const float* v = red + ((r * quads_per_wave + q) * 9 + k) * 4;
      s0 += (double)v[0];
      s1 += (double)v[1];
      s2 += (double)v[2];
      s3 += (double)v[3];
    }
    double* out = partial + ((int64_t)blockIdx.y * 9 + k) * ci.in_c + c;
    out[0] = s0;
    out[1] = s1;
    out[2] = s2;
    out[3] = s3;
  }
}

// Position (row-major over the dilated window) of the first strict maximum of the window of
// output pixel (yr, yc), as maxPoolPositions finds it; -1 when nothing is greater than -inf.
__device__ __forceinline__ int max_position(const float* x, const tfhip_conv2d_info& ci, int eff_h,
                                            int eff_w, int n, int yr, int yc, int d) {
  const int xr_corner = yr * ci.stride_h - ci.pad_top, xc_corner = yc * ci.stride_w - ci.pad_left;
  float best = -__builtin_inff();
  int pos = -1;
  for (int wr = 0; wr < eff_h; wr += ci.dilation_h) {
    const int xr = xr_corner + wr;
    if ((unsigned)xr >= (unsigned)ci.in_h) continue;
    for (int wc = 0; wc < eff_w; wc += ci.dilation_w) {
      const int xc = xc_corner + wc;
      if ((unsigned)xc >= (unsigned)ci.in_w) continue;
      const float v = x[(((int64_t)n * ci.in_h + xr) * ci.in_w + xc) * ci.in_c + d];
      if (v > best) {
        best = v;
        pos = wr * eff_w + wc;
      }
    }
  }
  return pos;
}

// One lane per dx element.  kind 1 (max): dy of every covering window whose first maximum is
// this pixel; kind 0 (avg): dy of every covering window times 1 / (filter_h * filter_w).
__global__ void pool2d_backprop_kernel(const float* dy, const float* x, float* dx,
                                       const tfhip_conv2d_info ci, int kind) {
  const int eff_h = ci.filter_h + (ci.filter_h - 1) * (ci.dilation_h - 1);
  const int eff_w = ci.filter_w + (ci.filter_w - 1) * (ci.dilation_w - 1);
  const int pad_top = eff_h - 1 - ci.pad_top, pad_left = eff_w - 1 - ci.pad_left;
  const double avg_multiplier = 1.0 / (double)(ci.filter_h * ci.filter_w);
  const int64_t total = (int64_t)ci.batch * ci.in_h * ci.in_w * ci.in_c;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += stride) {
    const int d = (int)(g % ci.in_c);
    int64_t t = g / ci.in_c;
    const int xc = (int)(t % ci.in_w);
    t /= ci.in_w;
    const int xr = (int)(t % ci.in_h);
    const int n = (int)(t / ci.in_h);
    const int dyr_corner = xr - pad_top, dyc_corner = xc - pad_left;
    double dot = 0.0;
    for (int wr = 0; wr < eff_h; wr += ci.dilation_h) {
      const int num_r = dyr_corner + wr;
      if (num_r < 0 || num_r % ci.stride_h != 0) continue;
      const int yr = num_r / ci.stride_h;
      if (yr >= ci.out_h) continue;
      for (int wc = 0; wc < eff_w; wc += ci.dilation_w) {
        const int num_c = dyc_corner + wc;
        if (num_c < 0 || num_c % ci.stride_w != 0) continue;
        const int yc = num_c / ci.stride_w;
        if (yc >= ci.out_w) continue;
        if (kind == TFHIP_POOL_MAX) {
          const int max_pos = eff_h * eff_w - 1 - max_position(x, ci, eff_h, eff_w, n, yr, yc, d);
          if (max_pos != wr * eff_w + wc) continue;
        }
        dot += (double)dy[(((int64_t)n * ci.out_h + yr) * ci.out_w + yc) * ci.out_c + d];
      }
    }
    dx[g] = (float)(kind == TFHIP_POOL_MAX ? dot : dot * avg_multiplier);
  }
}

// The same with a lane owning 4 consecutive channels (C % 4 == 0, 16-byte aligned buffers):
// the window scan and the dy gather are 16-byte accesses, the winner is tracked per channel.
__global__ __launch_bounds__(256) void pool2d_backprop_vec_kernel(
    const float* __restrict__ dy, const float* __restrict__ x, float* __restrict__ dx,
    const tfhip_conv2d_info ci, int kind, uint32_t total, Divisor by_c4, Divisor by_w, Divisor by_h,
    Divisor by_sh, Divisor by_sw) {
  const int eff_h = ci.filter_h + (ci.filter_h - 1) * (ci.dilation_h - 1);
  const int eff_w = ci.filter_w + (ci.filter_w - 1) * (ci.dilation_w - 1);
  const int pad_top = eff_h - 1 - ci.pad_top, pad_left = eff_w - 1 - ci.pad_left;
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= total) return;
  uint32_t t = g;
  const int cq = (int)by_c4.divmod(t), xc = (int)by_w.divmod(t), xr = (int)by_h.divmod(t), n = (int)t;
  const float* xn = x + (int64_t)n * ci.in_h * ci.in_w * ci.in_c + cq * 4;
  const float* dyn = dy + (int64_t)n * ci.out_h * ci.out_w * ci.out_c + cq * 4;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int wr = 0; wr < eff_h; wr += ci.dilation_h) {
    const int num_r = xr - pad_top + wr;
    const int yr = (int)by_sh.quotient((uint32_t)max(num_r, 0));
    if (num_r < 0 || yr * ci.stride_h != num_r || yr >= ci.out_h) continue;
    for (int wc = 0; wc < eff_w; wc += ci.dilation_w) {
      const int num_c = xc - pad_left + wc;
      const int yc = (int)by_sw.quotient((uint32_t)max(num_c, 0));
      if (num_c < 0 || yc * ci.stride_w != num_c || yc >= ci.out_w) continue;
      const f32x4 d = *reinterpret_cast<const f32x4*>(dyn + ((int64_t)yr * ci.out_w + yc) * ci.out_c);
      if (kind != TFHIP_POOL_MAX) {
        acc += d;
        continue;
      }
      // first strict maximum of window (yr, yc), per channel; this pixel sits at the
      // flipped position (eff_h - 1 - wr, eff_w - 1 - wc) of that window
      const int xr0 = yr * ci.stride_h - ci.pad_top, xc0 = yc * ci.stride_w - ci.pad_left;
      f32x4 best = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
      int pos[4] = {-1, -1, -1, -1};
      for (int fr = 0; fr < eff_h; fr += ci.dilation_h) {
        const int r = xr0 + fr;
        if ((unsigned)r >= (unsigned)ci.in_h) continue;
        for (int fc = 0; fc < eff_w; fc += ci.dilation_w) {
          const int c = xc0 + fc;
          if ((unsigned)c >= (unsigned)ci.in_w) continue;
          const f32x4 v = *reinterpret_cast<const f32x4*>(xn + ((int64_t)r * ci.in_w + c) * ci.in_c);
#pragma unroll
          for (int e = 0; e < 4; e++)
            if (v[e] > best[e]) {
              best[e] = v[e];
              pos[e] = fr * eff_w + fc;
            }
        }
      }
      const int mine = (eff_h - 1 - wr) * eff_w + (eff_w - 1 - wc);
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (pos[e] == mine) acc[e] += d[e];
    }
  }
  if (kind != TFHIP_POOL_MAX) acc *= 1.0f / (float)(ci.filter_h * ci.filter_w);
  *reinterpret_cast<f32x4*>(dx + (int64_t)g * 4) = acc;
}

// maxPoolBackprop of F x F windows at stride S <= F (no dilation): a lane owns the S x S pixels that
// start where window (by, bx) starts, for 4 channels.  It reads what the M x M windows over them see
// once, finds every window's winner, and stores its pixels.  Bound by memory: [32,56,56,128], 2 x 2 at
// stride 2, 17.9 us (6.4 TB/s), 3 x 3 36.5.  One lane per pixel (pool2d_backprop_vec_kernel) scans every window
// once per pixel it covers, 39.5 and 124.5 us.
// Pixels beyond the image read as -inf, which never wins; a pixel's gradients are added window row
// by window row, as there.
template <int F, int S>
__global__ __launch_bounds__(256) void max_pool_backprop_block_kernel(
    const float* __restrict__ dy, const float* __restrict__ x, float* __restrict__ dx,
    const tfhip_conv2d_info ci, uint32_t total, Divisor by_c4, Divisor by_bw, Divisor by_bh) {
  constexpr int M = (F + S - 1) / S;      // windows over a block, per direction
  constexpr int R = (M - 1) * S + F;      // rows (columns) of x that they see
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= total) return;
  uint32_t t = g;
  const int cq = (int)by_c4.divmod(t), bx = (int)by_bw.divmod(t), by = (int)by_bh.divmod(t), n = (int)t;
  const int r0 = (by - (M - 1)) * S - ci.pad_top, c0 = (bx - (M - 1)) * S - ci.pad_left;
  const int64_t image = (int64_t)n * ci.in_h * ci.in_w * ci.in_c + cq * 4;
  const float* xn = x + image;
  const float* dyn = dy + (int64_t)n * ci.out_h * ci.out_w * ci.out_c + cq * 4;
  const f32x4 none = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
  f32x4 v[R][R], d[M][M];
#pragma unroll
  for (int i = 0; i < R; i++)
#pragma unroll
    for (int j = 0; j < R; j++) {
      const int r = min(max(r0 + i, 0), ci.in_h - 1), c = min(max(c0 + j, 0), ci.in_w - 1);
      v[i][j] = *reinterpret_cast<const f32x4*>(xn + ((int64_t)r * ci.in_w + c) * ci.in_c);
    }
#pragma unroll
  for (int a = 0; a < M; a++)
#pragma unroll
    for (int b = 0; b < M; b++) {
      const int yr = min(max(by - (M - 1) + a, 0), ci.out_h - 1), yc = min(max(bx - (M - 1) + b, 0), ci.out_w - 1);
      d[a][b] = *reinterpret_cast<const f32x4*>(dyn + ((int64_t)yr * ci.out_w + yc) * ci.out_c);
    }
#pragma unroll
  for (int i = 0; i < R; i++)
#pragma unroll
    for (int j = 0; j < R; j++)
      if ((unsigned)(r0 + i) >= (unsigned)ci.in_h || (unsigned)(c0 + j) >= (unsigned)ci.in_w) v[i][j] = none;
  f32x4 acc[S][S];
#pragma unroll
  for (int i = 0; i < S; i++)
#pragma unroll
    for (int j = 0; j < S; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int a = 0; a < M; a++)
#pragma unroll
    for (int b = 0; b < M; b++) {
      // the window's first strict maximum; -1: no pixel, or no window here
      const bool there = (unsigned)(by - (M - 1) + a) < (unsigned)ci.out_h &&
                         (unsigned)(bx - (M - 1) + b) < (unsigned)ci.out_w;
      f32x4 best = none;
      int pos[4] = {-1, -1, -1, -1};
#pragma unroll
      for (int i = 0; i < F; i++)
#pragma unroll
        for (int j = 0; j < F; j++)
#pragma unroll
          for (int e = 0; e < 4; e++)
            if (v[a * S + i][b * S + j][e] > best[e]) {
              best[e] = v[a * S + i][b * S + j][e];
              pos[e] = i * F + j;
            }
#pragma unroll
      for (int i = 0; i < S; i++)
#pragma unroll
        for (int j = 0; j < S; j++) {
          const int wi = (M - 1 - a) * S + i, wj = (M - 1 - b) * S + j;  // this pixel in that window
          if (wi >= F || wj >= F) continue;
#pragma unroll
          for (int e = 0; e < 4; e++) acc[i][j][e] += there && pos[e] == wi * F + wj ? d[a][b][e] : 0.f;
        }
    }
#pragma unroll
  for (int i = 0; i < S; i++)
#pragma unroll
    for (int j = 0; j < S; j++) {
      const int r = by * S - ci.pad_top + i, c = bx * S - ci.pad_left + j;
      if ((unsigned)r < (unsigned)ci.in_h && (unsigned)c < (unsigned)ci.in_w)
        *reinterpret_cast<f32x4*>(dx + image + ((int64_t)r * ci.in_w + c) * ci.in_c) = acc[i][j];
    }
}

static int check_geometry(tfhip_ctx* ctx, const char* op, const tfhip_conv2d_info* ci,
                          bool dilation_allowed) {
  if (ci->batch < 0 || ci->in_h < 0 || ci->in_w < 0 || ci->in_c < 0 || ci->out_h < 0 ||
      ci->out_w < 0 || ci->out_c < 0 || ci->filter_h <= 0 || ci->filter_w <= 0 ||
      ci->stride_h <= 0 || ci->stride_w <= 0 || ci->dilation_h <= 0 || ci->dilation_w <= 0)
    return ctx->fail(TFHIP_EINVAL, "%s: bad geometry", op);
  if (!dilation_allowed && (ci->dilation_h != 1 || ci->dilation_w != 1))
    return ctx->fail(TFHIP_EINVAL, "%s: dilation rates greater than 1 are not yet supported", op);
  return TFHIP_OK;
}

static int der_filter_finish(tfhip_ctx* ctx, const void* partial, const Buf* bdw, int64_t w_n, int64_t slices) {
  tfhip::launch(ctx, depthwise_der_filter_finish_kernel, dim3((unsigned)ceil_div(w_n, 32)), dim3(1024), 0,
                static_cast<const double*>(partial), static_cast<float*>(bdw->ptr), w_n, (int)slices);
  TFHIP_LAUNCH_CHECK_NAMED(ctx, "depthwise_der_filter_finish");
  return TFHIP_OK;
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

static unsigned grid_for(tfhip_ctx* ctx, int64_t elements) {
  const int64_t blocks = ceil_div(elements, 256);
  const int64_t cap = (int64_t)ctx->num_cus * 16;
  return (unsigned)(blocks > cap ? cap : blocks);
}

}  // namespace tfhip

using namespace tfhip;

extern "C" int tfhip_depthwise_conv2d_der_input(tfhip_ctx* ctx, int64_t dy, int64_t filter,
                                                int64_t dx, const tfhip_conv2d_info* ci) {
  if (!ctx || !ci) return TFHIP_EINVAL;
  int rc;
  if ((rc = check_geometry(ctx, "depthwiseConv2DDerInput", ci, false))) return rc;
  TFHIP_GET(ctx, bdy, dy);
  TFHIP_GET(ctx, bw, filter);
  TFHIP_GET(ctx, bdx, dx);
  if (ci->in_c <= 0 || ci->out_c % ci->in_c != 0)
    return ctx->fail(TFHIP_EINVAL, "depthwiseConv2DDerInput: out channels must be a multiple of in channels");
  const int ch_mul = ci->out_c / ci->in_c;
  const int64_t x_n = (int64_t)ci->batch * ci->in_h * ci->in_w * ci->in_c;
  const int64_t w_n = (int64_t)ci->filter_h * ci->filter_w * ci->out_c;
  const int64_t y_n = (int64_t)ci->batch * ci->out_h * ci->out_w * ci->out_c;
  if (bdy->numel != y_n || bw->numel != w_n || bdx->numel != x_n)
    return ctx->fail(TFHIP_EINVAL, "depthwiseConv2DDerInput: buffer sizes do not match the geometry");
  if (bdx->dtype != TFHIP_FLOAT32 || bw->dtype == TFHIP_UINT8Q)
    return ctx->fail(TFHIP_EINVAL, "depthwiseConv2DDerInput: dx must be float32 and the filter not quantised");
  if (x_n == 0) return TFHIP_OK;
  Temp tdy(ctx), tw(ctx);
  const float *dyf, *wf;
  if ((rc = as_f32(ctx, bdy, &tdy, &dyf))) return rc;
  if ((rc = as_f32(ctx, bw, &tw, &wf))) return rc;
  float* dxf = static_cast<float*>(bdx->ptr);
  if (ch_mul == 1 && ci->stride_h == 1 && ci->stride_w == 1 && y_n > 0) {
    // stride 1: dx is the depthwise convolution of dy with the filter flipped in both spatial
    // directions and the padding filter - 1 - pad: the forward kernels do it at their speed
    tfhip_conv2d_info back = *ci;
    back.in_h = ci->out_h; back.in_w = ci->out_w;
    back.out_h = ci->in_h; back.out_w = ci->in_w;
    back.out_c = ci->in_c;
    back.pad_top = ci->filter_h - 1 - ci->pad_top;
    back.pad_left = ci->filter_w - 1 - ci->pad_left;
    back.pad_bottom = back.pad_right = 0;   // (not read by the kernels)
    if ((rc = depthwise_mirrored_f32(ctx, dyf, wf, dxf, &back))) return rc;
    strncat(ctx->last_kernel, "_as_der_input", sizeof ctx->last_kernel - strlen(ctx->last_kernel) - 1);
    return TFHIP_OK;
  }
  if (ch_mul == 1 && ci->in_c % 4 == 0 && x_n / 4 <= INDEX32 - 256 && aligned16(dyf) && aligned16(wf) &&
      aligned16(dxf)) {
    const unsigned blocks = (unsigned)ceil_div(x_n / 4, 256);
    const int s = ci->stride_h == ci->stride_w && ci->stride_h <= 2 ? ci->stride_h : 0;
    ctx->name_kernel("depthwise_der_input_vec_s%d", s);
    if (s == 1)
      tfhip::launch(ctx, depthwise_der_input_vec_kernel<1>, dim3(blocks), dim3(256), 0,
                         dyf, wf, dxf, *ci, (uint32_t)(x_n / 4), Divisor(ci->in_c / 4),
                         Divisor(ci->in_w), Divisor(ci->in_h));
    else if (s == 2)
      tfhip::launch(ctx, depthwise_der_input_vec_kernel<2>, dim3(blocks), dim3(256), 0,
                         dyf, wf, dxf, *ci, (uint32_t)(x_n / 4), Divisor(ci->in_c / 4),
                         Divisor(ci->in_w), Divisor(ci->in_h));
    else
      tfhip::launch(ctx, depthwise_der_input_vec_kernel<0>, dim3(blocks), dim3(256), 0,
                         dyf, wf, dxf, *ci, (uint32_t)(x_n / 4), Divisor(ci->in_c / 4),
                         Divisor(ci->in_w), Divisor(ci->in_h));
    TFHIP_LAUNCH_CHECK(ctx);
    return TFHIP_OK;
  }
  ctx->name_kernel("depthwise_der_input");
  tfhip::launch(ctx, depthwise_der_input_kernel, dim3(grid_for(ctx, x_n)), dim3(256), 0,
                     dyf, wf, dxf, *ci, ch_mul);
  TFHIP_LAUNCH_CHECK(ctx);
  return TFHIP_OK;
}

extern "C" int tfhip_depthwise_conv2d_der_filter(tfhip_ctx* ctx, int64_t x, int64_t dy, int64_t dw,
                                                 const tfhip_conv2d_info* ci) {
  if (!ctx || !ci) return TFHIP_EINVAL;
  int rc;
  if ((rc = check_geometry(ctx, "depthwiseConv2DDerFilter", ci, false))) return rc;
  TFHIP_GET(ctx, bx, x);
  TFHIP_GET(ctx, bdy, dy);
  TFHIP_GET(ctx, bdw, dw);
  if (ci->in_c <= 0 || ci->out_c % ci->in_c != 0)
    return ctx->fail(TFHIP_EINVAL, "depthwiseConv2DDerFilter: out channels must be a multiple of in channels");
  const int ch_mul = ci->out_c / ci->in_c;
  const int64_t x_n = (int64_t)ci->batch * ci->in_h * ci->in_w * ci->in_c;
  const int64_t w_n = (int64_t)ci->filter_h * ci->filter_w * ci->out_c;
  const int64_t y_n = (int64_t)ci->batch * ci->out_h * ci->out_w * ci->out_c;
  if (bx->numel != x_n || bdy->numel != y_n || bdw->numel != w_n)
    return ctx->fail(TFHIP_EINVAL, "depthwiseConv2DDerFilter: buffer sizes do not match the geometry");
  if (bdw->dtype != TFHIP_FLOAT32)
    return ctx->fail(TFHIP_EINVAL, "depthwiseConv2DDerFilter: dW must be float32");
  if (w_n == 0) return TFHIP_OK;
  const int taps = ci->filter_h * ci->filter_w;
  if (taps > 65535) return ctx->fail(TFHIP_ENOTSUP, "depthwiseConv2DDerFilter: more than 65535 filter taps");
  Temp tx(ctx), tdy(ctx), tpart(ctx);
  const float *xf, *dyf;
  if ((rc = as_f32(ctx, bx, &tx, &xf))) return rc;
  if ((rc = as_f32(ctx, bdy, &tdy, &dyf))) return rc;
  const int64_t pixels = (int64_t)ci->batch * ci->out_h * ci->out_w;
  // (buffer descriptors: both operands below 2 GiB)
  if (ch_mul == 1 && ci->filter_h == 3 && ci->filter_w == 3 && ci->in_c % 4 == 0 && aligned16(xf) &&
      aligned16(dyf) && pixels > 0 && x_n > 0 && x_n < (1 << 29) && y_n < (1 << 29) &&
      ci->stride_h == ci->stride_w && ci->stride_h <= 2) {
    const int c4 = ci->in_c / 4;
    int qpw = 1;                       // channel quads per workgroup: a power of two <= 64
    while (qpw < 64 && qpw < c4) qpw *= 2;
    const int64_t blocks_c = ceil_div(c4, qpw);
    const int subs = 256 / qpw;
    // The columns of the output are cut into segments until four workgroups per CU, which is what their LDS
    // allows, have one each.  A segment reads two rows of x more than it has, so it is made no shorter
    // than its chain of float32 additions may be long: 8, or what dealing the pixels evenly over
    // workgroups of 8 pixels a lane gives.  (Segments of at least 8 rows, 14 where the image has 14:
    // [8, 14, 14, 512] 6.0 us and 7.2e-8 from the sum in 64 bits, 5.5 us and 5.5e-8 in halves; [1, 14, 14, 512]
    // 5.9 and 4.7; [16, 28, 28, 256] 9.2 and 9.4; [64, 28, 28, 256] at stride 2 13.7 and 14.3, 7.3e-8 and 5.6e-8.)
    const int64_t columns = (int64_t)ci->batch * ci->out_w, most = ceil_div((int64_t)ctx->num_cus * 4, blocks_c);
    const int64_t chain = ceil_div(ceil_div(pixels, ceil_div(pixels, (int64_t)subs * 8)), subs);
    int64_t segs = std::max<int64_t>(1, std::min<int64_t>(most * subs / columns, ceil_div(ci->out_h, chain)));
    const int64_t rows = ceil_div(ci->out_h, segs);
    segs = ceil_div(ci->out_h, rows);
    const int64_t units = columns * segs, per_lane = ceil_div(units, most * subs);
    const int64_t slices = ceil_div(units, per_lane * subs);
    if (!tpart.get((size_t)(slices * w_n) * sizeof(double))) return TFHIP_EDEVICE;
    ctx->name_kernel("depthwise3x3_der_filter");
    tfhip::launch(ctx, ci->stride_h == 1 ? depthwise3x3_der_filter_rows_kernel<1> : depthwise3x3_der_filter_rows_kernel<2>,
                  dim3((unsigned)blocks_c, (unsigned)slices), dim3(256), (size_t)(256 * 9 * 4 * sizeof(float)), xf, dyf,
                  static_cast<double*>(tpart.ptr), *ci, (unsigned)(x_n * 4), (unsigned)(y_n * 4), qpw, (int)rows,
                  (uint32_t)units, Divisor(ci->out_w), Divisor(segs));
    TFHIP_LAUNCH_CHECK(ctx);
    return der_filter_finish(ctx, tpart.ptr, bdw, w_n, slices);
  }
  if (ch_mul == 1 && ci->filter_h == 3 && ci->filter_w == 3 && ci->in_c % 4 == 0 && aligned16(xf) &&
      aligned16(dyf) && pixels > 0 && pixels <= INDEX32) {
    const int c4 = ci->in_c / 4;
    int qpw = 1;                       // channel quads per workgroup: a power of two <= 64
    while (qpw < 64 && qpw < c4) qpw *= 2;
    const int64_t blocks_c = ceil_div(c4, qpw);
    const int subs = 256 / qpw;
    // two workgroups per CU, and at least 8 pixels per lane.  A lane's pixels are a chain of loads
    // of about 0.8 us each, which a layer with fewer of them is bound by: [8, 14, 14, 512] 25.4 us
    // with at least 32 pixels, 12.8 with 8 (16.9 with 16); [64, 28, 28, 256] stride 2 32.9 -> 19.8,
    // [32, 56, 56, 128] 39.0 -> 36.6 (40.0 with four workgroups per CU: more partial sums).
    int64_t slices = ceil_div((int64_t)ctx->num_cus * 2, blocks_c);
    if (slices > ceil_div(pixels, (int64_t)subs * 8)) slices = ceil_div(pixels, (int64_t)subs * 8);
    if (slices < 1) slices = 1;
    if (slices > 65535) slices = 65535;
    const int64_t per_slice = ceil_div(pixels, slices);
    if (!tpart.get((size_t)(slices * w_n) * sizeof(double))) return TFHIP_EDEVICE;
    ctx->name_kernel("depthwise3x3_der_filter");
    tfhip::launch(ctx, depthwise3x3_der_filter_partial_kernel, dim3((unsigned)blocks_c, (unsigned)slices),
                       dim3(256), (size_t)(256 * 9 * 4 * sizeof(float)), xf, dyf,
                       static_cast<double*>(tpart.ptr), *ci, qpw, per_slice, Divisor(ci->out_w), Divisor(ci->out_h));
    TFHIP_LAUNCH_CHECK(ctx);
    return der_filter_finish(ctx, tpart.ptr, bdw, w_n, slices);
  }
  // enough pixel slices to fill the machine, at least 64 pixels each
  const int64_t channel_blocks = ceil_div(ci->out_c, 64);
  int64_t slices = ceil_div((int64_t)ctx->num_cus * 8, channel_blocks * taps);
  if (slices > ceil_div(pixels, 64)) slices = ceil_div(pixels, 64);
  if (slices < 1) slices = 1;
  if (slices > 65535) slices = 65535;
  const int64_t per_slice = ceil_div(pixels > 0 ? pixels : 1, slices);
  if (!tpart.get((size_t)(slices * w_n) * sizeof(double))) return TFHIP_EDEVICE;
  ctx->name_kernel("depthwise_der_filter");
  tfhip::launch(ctx, depthwise_der_filter_partial_kernel,
                     dim3((unsigned)channel_blocks, (unsigned)taps, (unsigned)slices), dim3(256), 0, xf, dyf, static_cast<double*>(tpart.ptr), *ci, ch_mul, per_slice);
  TFHIP_LAUNCH_CHECK(ctx);
  return der_filter_finish(ctx, tpart.ptr, bdw, w_n, slices);
}

extern "C" int tfhip_pool2d_backprop(tfhip_ctx* ctx, int64_t dy, int64_t x, int64_t dx,
                                     const tfhip_conv2d_info* ci, int kind) {
  if (!ctx || !ci) return TFHIP_EINVAL;
  int rc;
  if ((rc = check_geometry(ctx, "poolBackprop", ci, true))) return rc;
  if (kind != TFHIP_POOL_AVG && kind != TFHIP_POOL_MAX)
    return ctx->fail(TFHIP_EINVAL, "poolBackprop: unknown kind %d", kind);
  TFHIP_GET(ctx, bdy, dy);
  TFHIP_GET(ctx, bx, x);
  TFHIP_GET(ctx, bdx, dx);
  if (ci->in_c != ci->out_c) return ctx->fail(TFHIP_EINVAL, "poolBackprop: channel counts differ");
  const int64_t x_n = (int64_t)ci->batch * ci->in_h * ci->in_w * ci->in_c;
  const int64_t y_n = (int64_t)ci->batch * ci->out_h * ci->out_w * ci->out_c;
  if (bdy->numel != y_n || bx->numel != x_n || bdx->numel != x_n)
    return ctx->fail(TFHIP_EINVAL, "poolBackprop: buffer sizes do not match the geometry");
  if (bdx->dtype != TFHIP_FLOAT32) return ctx->fail(TFHIP_EINVAL, "poolBackprop: dx must be float32");
  if (x_n == 0) return TFHIP_OK;
  Temp tdy(ctx), tx(ctx);
  const float *dyf, *xf;
  if ((rc = as_f32(ctx, bdy, &tdy, &dyf))) return rc;
  if ((rc = as_f32(ctx, bx, &tx, &xf))) return rc;
  float* dxf = static_cast<float*>(bdx->ptr);
  const bool vec = ci->in_c % 4 == 0 && x_n / 4 <= INDEX32 - 256 && aligned16(dyf) && aligned16(xf) && aligned16(dxf);
  // The windows that networks use: 2 x 2 and 3 x 3 at stride 2 (blocks outside the image's own
  // pixels exist on the padded side only).  y_n is 0 only where there is no window at all.
  const int f = ci->filter_h;
  if (vec && kind == TFHIP_POOL_MAX && y_n > 0 && ci->filter_w == f && (f == 2 || f == 3) && ci->stride_h == 2 &&
      ci->stride_w == 2 && ci->dilation_h == 1 && ci->dilation_w == 1 && ci->pad_top >= 0 && ci->pad_left >= 0 &&
      ci->pad_top < f && ci->pad_left < f) {
    const int64_t bh = (ci->in_h - 1 + ci->pad_top) / 2 + 1, bw = (ci->in_w - 1 + ci->pad_left) / 2 + 1;
    const int64_t total = (int64_t)ci->batch * bh * bw * (ci->in_c / 4);
    if (total <= INDEX32 - 256) {
      ctx->name_kernel("max_pool_backprop_%dx%d_s2", f, f);
      tfhip::launch(ctx, f == 2 ? max_pool_backprop_block_kernel<2, 2> : max_pool_backprop_block_kernel<3, 2>,
                    dim3((unsigned)ceil_div(total, 256)), dim3(256), 0, dyf, xf, dxf, *ci, (uint32_t)total,
                    Divisor(ci->in_c / 4), Divisor(bw), Divisor(bh));
      TFHIP_LAUNCH_CHECK(ctx);
      return TFHIP_OK;
    }
  }
  if (vec) {
    ctx->name_kernel(
             kind == TFHIP_POOL_MAX ? "max_pool_backprop_vec" : "avg_pool_backprop_vec");
    tfhip::launch(ctx, pool2d_backprop_vec_kernel, dim3((unsigned)ceil_div(x_n / 4, 256)), dim3(256), 0, dyf, xf, dxf, *ci, kind,
                  (uint32_t)(x_n / 4), Divisor(ci->in_c / 4), Divisor(ci->in_w), Divisor(ci->in_h),
                  Divisor(ci->stride_h), Divisor(ci->stride_w));
    TFHIP_LAUNCH_CHECK(ctx);
    return TFHIP_OK;
  }
  ctx->name_kernel(
           kind == TFHIP_POOL_MAX ? "max_pool_backprop" : "avg_pool_backprop");
  tfhip::launch(ctx, pool2d_backprop_kernel, dim3(grid_for(ctx, x_n)), dim3(256), 0, dyf,
                     xf, static_cast<float*>(bdx->ptr), *ci, kind);
  TFHIP_LAUNCH_CHECK(ctx);
  return TFHIP_OK;
}
