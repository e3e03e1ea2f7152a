// Data-movement and pointwise kernels that converter graphs use around the convolutions:
// a strided box copy (slice, stridedSlice, reverse, concat, pad, tile), logicalNot,
// batchNormalization, resizeBilinear, oneHot.  Replaces backend_cpu.ts:292-433, 795-804,
// 2152-2176, 2875-2936, 3167-3213, 3325-3339 of the reference.  All of them stream HBM
// once; the innermost dimension of the box runs along the lanes.
#include "tfhip_internal.h"

namespace tfhip {

constexpr int MAXBOX = 8;
struct BoxArgs {
  int rank;
  int region[MAXBOX];
  int64_t x_stride[MAXBOX], out_stride[MAXBOX];
  int64_t x_offset, out_offset;
};

template <typename T>
__global__ void strided_copy_kernel(const T* __restrict__ x, T* __restrict__ out, int64_t n,
                                    BoxArgs b) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    int64_t rem = i, src = b.x_offset, dst = b.out_offset;
#pragma unroll
    for (int d = MAXBOX - 1; d >= 0; d--) {
      if (d < b.rank) {
        const int64_t c = rem % b.region[d];
        rem /= b.region[d];
        src += c * b.x_stride[d];
        dst += c * b.out_stride[d];
      }
    }
    out[dst] = x[src];
  }
}

// The same where every index fits 32 bits, over the dimensions that are left when those that run
// on into each other on both sides are one.  Four elements in flight per lane.  Mirroring
// [16, 480, 640, 3]: 65 us with 64-bit divisions by the four extents, 21.7 with these.
struct Box32 {
  int rank;
  int32_t x_offset, out_offset;
  Divisor region[MAXBOX];
  int32_t x_stride[MAXBOX], out_stride[MAXBOX];
};
// The same for boxes of runs: 4-byte elements that lie side by side on both sides (the innermost
// dimension, which `outer` does not hold), copied in vectors of 4 at 4-byte alignment, which the
// hardware takes.  MIRROR = 0: runs of `len` elements.  MIRROR = 1 .. 3: rows of `len` elements in pixels
// of so many, read backwards pixel by pixel; the four elements of a vector come from one line or two.
// What the end of a row cuts is copied as a whole vector too, from before the end, the same values
// twice.  Mirroring [16, 480, 640, 3] left to right 22.2 -> 18.5 us (6.4 TB/s), top to bottom 20.0 -> 18.0;
// placing [32, 56, 56, 64] in the channels of a larger tensor 10.6 -> 8.8.
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
struct __attribute__((packed, aligned(4))) Loose4 {
  i32x4 v;
};
template <int MIRROR>
__global__ __launch_bounds__(256) void copy_runs_kernel(const int32_t* __restrict__ x, int32_t* __restrict__ out,
                                                        uint32_t n, Box32 outer, Divisor groups, int len) {
  constexpr int W = MIRROR ? MIRROR : 1;  // elements of a pixel
  uint32_t rem = blockIdx.x * blockDim.x + threadIdx.x;
  if (rem >= n) return;
  const int e0 = min((int)groups.divmod(rem) * 4, len - 4);
  int32_t src = outer.x_offset, dst = outer.out_offset + e0;
#pragma unroll
  for (int d = MAXBOX - 1; d >= 0; d--) {
    if (d < outer.rank) {
      const int32_t c = (int32_t)outer.region[d].divmod(rem);
      src += c * outer.x_stride[d];
      dst += c * outer.out_stride[d];
    }
  }
  i32x4 v;
  if (MIRROR == 0) {
    v = reinterpret_cast<const Loose4*>(x + src + e0)->v;
  } else if (MIRROR == 1) {  // (x_offset is the row's last element)
    const i32x4 t = reinterpret_cast<const Loose4*>(x + src - e0 - 3)->v;
    v = i32x4{t[3], t[2], t[1], t[0]};
  } else {                   // (x_offset is the row's last pixel)
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = x[src - (e0 + e) / W * W + (e0 + e) % W];
  }
  reinterpret_cast<Loose4*>(out + dst)->v = v;
}

template <typename T>
__global__ void strided_copy32_kernel(const T* __restrict__ x, T* __restrict__ out, uint32_t n, Box32 b) {
  constexpr int U = 4;
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i0 = blockIdx.x * blockDim.x + threadIdx.x; i0 < n; i0 += U * stride) {
    int32_t src[U], dst[U];
    uint32_t rem[U];
    T v[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      rem[u] = i0 + u * stride;
      src[u] = b.x_offset;
      dst[u] = b.out_offset;
    }
#pragma unroll
    for (int d = MAXBOX - 1; d >= 0; d--) {
      if (d < b.rank) {
#pragma unroll
        for (int u = 0; u < U; u++) {
          const int32_t c = (int32_t)b.region[d].divmod(rem[u]);
          src[u] += c * b.x_stride[d];
          dst[u] += c * b.out_stride[d];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++)
      if (i0 + u * stride < n) v[u] = x[src[u]];
#pragma unroll
    for (int u = 0; u < U; u++)
      if (i0 + u * stride < n) out[dst[u]] = v[u];
  }
}

__global__ void logical_not_kernel(const uint8_t* x, uint8_t* out, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    out[i] = x[i] ? 0 : 1;
}

// The reference evaluates offset + (x - mean) * scale / sqrt(variance + eps) in double and
// rounds once at the store; float32 arithmetic here stays within 1e-6 relative of that.
__global__ void batchnorm_kernel(const float* x, const float* mean, int64_t n_mean,
                                 const float* variance, int64_t n_var, const float* offset,
                                 int64_t n_off, const float* scale, int64_t n_scale, float eps,
                                 float* out, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const float m = mean[i % n_mean], v = variance[i % n_var];
    const float s = scale ? scale[i % n_scale] : 1.f;
    const float o = offset ? offset[i % n_off] : 0.f;
    out[i] = o + (x[i] - m) * s / sqrtf(v + eps);
  }
}

// The same over [rows, C] with every operand given per channel: the statistics of four channels in
// 16-byte accesses.  Bound by HBM: [100352, 128] 42 us with four 64-bit remainders per element,
// 18.0 with one per four.
typedef float bn_f32x4 __attribute__((ext_vector_type(4)));
__global__ void batchnorm_channels_kernel(const bn_f32x4* __restrict__ x, const bn_f32x4* __restrict__ mean,
                                          const bn_f32x4* __restrict__ variance,
                                          const bn_f32x4* __restrict__ offset,
                                          const bn_f32x4* __restrict__ scale, float eps,
                                          bn_f32x4* __restrict__ out, uint32_t n4, Divisor c4) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += stride) {
    uint32_t q = i;
    const uint32_t c = c4.divmod(q);
    const bn_f32x4 v = x[i], m = mean[c], var = variance[c];
    const bn_f32x4 s = scale ? scale[c] : bn_f32x4{1.f, 1.f, 1.f, 1.f};
    const bn_f32x4 o = offset ? offset[c] : bn_f32x4{0.f, 0.f, 0.f, 0.f};
    bn_f32x4 r;
#pragma unroll
    for (int e = 0; e < 4; e++) r[e] = o[e] + (v[e] - m[e]) * s[e] / sqrtf(var[e] + eps);
    out[i] = r;
  }
}

// One lane per output element, channel fastest.  Source coordinates as the reference
// computes them: ratio = effective input size / effective output size, floor / ceil
// neighbours, ceil clamped to the last row / column.
__global__ void resize_bilinear_kernel(const float* x, float* out, int batch, int in_h, int in_w,
                                       int ch, int out_h, int out_w, double ratio_h,
                                       double ratio_w) {
  const int64_t n = (int64_t)batch * out_h * out_w * ch;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const int d = (int)(i % ch);
    int64_t t = i / ch;
    const int c = (int)(t % out_w);
    t /= out_w;
    const int r = (int)(t % out_h);
    const int b = (int)(t / out_h);
    // double throughout, like the reference: a float product can land on the other side of
    // an integer and pick different neighbours
    const double fr = ratio_h * r, fc = ratio_w * c;
    const int r0 = (int)floor(fr), c0 = (int)floor(fc);
    const int r1 = min(in_h - 1, (int)ceil(fr)), c1 = min(in_w - 1, (int)ceil(fc));
    const double wr = fr - r0, wc = fc - c0;
    const float* xb = x + (int64_t)b * in_h * in_w * ch + d;
    const double tl = xb[((int64_t)r0 * in_w + c0) * ch], tr = xb[((int64_t)r0 * in_w + c1) * ch];
    const double bl = xb[((int64_t)r1 * in_w + c0) * ch], br = xb[((int64_t)r1 * in_w + c1) * ch];
    const double top = tl + (tr - tl) * wc;
    const double bot = bl + (br - bl) * wc;
    out[i] = (float)(top + (bot - top) * wr);
  }
}

// Nearest neighbour: source row / column = min(in - 1, floor(ratio * r)), or round half up
// (JavaScript's Math.round) with align_corners, in double as the reference computes them.
__global__ void resize_nearest_kernel(const float* x, float* out, int batch, int in_h, int in_w,
                                      int ch, int out_h, int out_w, double ratio_h,
                                      double ratio_w, int align_corners) {
  const int64_t n = (int64_t)batch * out_h * out_w * ch;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const int d = (int)(i % ch);
    int64_t t = i / ch;
    const int c = (int)(t % out_w);
    t /= out_w;
    const int r = (int)(t % out_h);
    const int b = (int)(t / out_h);
    const double fr = ratio_h * r, fc = ratio_w * c;
    const int sr = min(in_h - 1, (int)(align_corners ? floor(fr + 0.5) : floor(fr)));
    const int sc = min(in_w - 1, (int)(align_corners ? floor(fc + 0.5) : floor(fc)));
    out[i] = x[(((int64_t)b * in_h + sr) * in_w + sc) * ch + d];
  }
}

// The same with every index in 32 bits.  VEC = 4: four channels per lane in 16-byte accesses, where
// channels and pointers divide; VEC = 1 otherwise.  The three 64-bit divisions per element bounded both:
// bilinear [16, 480, 640, 3] -> 224 x 224 14.8 -> 10.8 us, [8, 224, 224, 3] -> 480 x 640 36.1 -> 18.3,
// [32, 56, 56, 64] -> 112 x 112 (128 MB in and out) 112 -> 30.9; nearest 10.6 -> 7.0, 27.0 -> 12.8, 82.2 -> 22.8.
template <int VEC>
struct Channels;
template <>
struct Channels<1> {
  typedef float T;
  static __device__ __forceinline__ float at(float v, int) { return v; }
  static __device__ __forceinline__ void put(float& v, int, float e) { v = e; }
};
template <>
struct Channels<4> {
  typedef float T __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ float at(const T& v, int e) { return v[e]; }
  static __device__ __forceinline__ void put(T& v, int e, float f) { v[e] = f; }
};
struct ResizePlan {
  uint32_t n;               // lanes: output elements / VEC
  Divisor ch, out_w, out_h;  // ch: channels / VEC
  int in_h, in_w;
  double ratio_h, ratio_w;
};
template <int VEC>
__global__ __launch_bounds__(256) void resize_bilinear32_kernel(const typename Channels<VEC>::T* __restrict__ x,
                                                                typename Channels<VEC>::T* __restrict__ out,
                                                                ResizePlan p) {
  typedef Channels<VEC> C;
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= p.n) return;
  uint32_t t = i;
  const uint32_t d = p.ch.divmod(t), c = p.out_w.divmod(t), r = p.out_h.divmod(t);
  const double fr = p.ratio_h * (int)r, fc = p.ratio_w * (int)c;
  const int r0 = (int)floor(fr), c0 = (int)floor(fc);
  const int r1 = min(p.in_h - 1, (int)ceil(fr)), c1 = min(p.in_w - 1, (int)ceil(fc));
  const double wr = fr - r0, wc = fc - c0;
  const uint32_t top_row = (t * p.in_h + r0) * p.in_w, bottom_row = (t * p.in_h + r1) * p.in_w;
  const auto tl4 = x[(top_row + c0) * p.ch.d + d], tr4 = x[(top_row + c1) * p.ch.d + d];
  const auto bl4 = x[(bottom_row + c0) * p.ch.d + d], br4 = x[(bottom_row + c1) * p.ch.d + d];
  typename C::T v;
#pragma unroll
  for (int e = 0; e < VEC; e++) {
    const double tl = C::at(tl4, e), tr = C::at(tr4, e), bl = C::at(bl4, e), br = C::at(br4, e);
    const double top = tl + (tr - tl) * wc;
    const double bot = bl + (br - bl) * wc;
    C::put(v, e, (float)(top + (bot - top) * wr));
  }
  out[i] = v;
}
template <int VEC>
__global__ __launch_bounds__(256) void resize_nearest32_kernel(const typename Channels<VEC>::T* __restrict__ x,
                                                               typename Channels<VEC>::T* __restrict__ out,
                                                               ResizePlan p, int align_corners) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= p.n) return;
  uint32_t t = i;
  const uint32_t d = p.ch.divmod(t), c = p.out_w.divmod(t), r = p.out_h.divmod(t);
  const double fr = p.ratio_h * (int)r, fc = p.ratio_w * (int)c;
  const int sr = min(p.in_h - 1, (int)(align_corners ? floor(fr + 0.5) : floor(fr)));
  const int sc = min(p.in_w - 1, (int)(align_corners ? floor(fc + 0.5) : floor(fc)));
  out[i] = x[((t * p.in_h + sr) * p.in_w + sc) * p.ch.d + d];
}
// Channels a lane takes, 0 where an index may pass 32 bits (the kernels above are for those).
int resize_width(const tfhip::Buf* x, const float* xf, const tfhip::Buf* out, int channels) {
  if (x->numel > INDEX32 || out->numel > INDEX32) return 0;
  return channels % 4 == 0 && !((reinterpret_cast<uintptr_t>(xf) | reinterpret_cast<uintptr_t>(out->ptr)) & 15) ? 4 : 1;
}
ResizePlan resize_plan(int64_t n, int vec, int channels, int in_h, int in_w, int out_h, int out_w, double ratio_h,
                       double ratio_w) {
  return ResizePlan{(uint32_t)(n / vec), Divisor(channels / vec), Divisor(out_w), Divisor(out_h), in_h, in_w,
                    ratio_h, ratio_w};
}

// out[i] = cond[i / inner] ? a[i] : b[i]; T = 4-byte (float32 / int32) or 1-byte (bool) elements.
template <typename T>
__global__ void select_kernel(const uint8_t* cond, const T* a, const T* b, T* out, int64_t n,
                              int64_t inner) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    out[i] = cond[i / inner] == 1 ? a[i] : b[i];
}

template <typename T>
__global__ void one_hot_kernel(const int32_t* idx, T* out, int64_t n_idx, int depth, T on, T off) {
  const int64_t n = n_idx * depth;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const int64_t e = i / depth;
    const int k = (int)(i - e * depth);
    out[i] = idx[e] == k ? on : off;
  }
}

static int grid_for(tfhip_ctx* ctx, int64_t work_items, int block) {
  const int64_t want = ceil_div(work_items, block);
  const int64_t cap = (int64_t)ctx->num_cus * 16;
  return (int)(want < 1 ? 1 : (want > cap ? cap : want));
}

}  // namespace tfhip

using namespace tfhip;

extern "C" int tfhip_strided_copy(tfhip_ctx* ctx, int64_t x, int64_t out, int rank,
                                  const int32_t* region, const int64_t* x_strides,
                                  int64_t x_offset, const int64_t* out_strides,
                                  int64_t out_offset) {
  if (!ctx) return TFHIP_EINVAL;
  if (rank < 0 || rank > MAXBOX) return ctx->fail(TFHIP_ENOTSUP, "strided copy: rank above %d", MAXBOX);
  if (rank > 0 && (!region || !x_strides || !out_strides)) return ctx->fail(TFHIP_EINVAL, "strided copy: null box");
  TFHIP_GET(ctx, bx, x);
  TFHIP_GET(ctx, bo, out);
  if (bx->dtype == TFHIP_UINT8Q || bo->dtype == TFHIP_UINT8Q || dtype_size(bx->dtype) != dtype_size(bo->dtype))
    return ctx->fail(TFHIP_EINVAL, "strided copy: source and destination element sizes differ");
  BoxArgs b = {};
  b.rank = rank;
  b.x_offset = x_offset;
  b.out_offset = out_offset;
  int64_t n = 1;
  // smallest and largest index the box touches on either side
  int64_t x_lo = x_offset, x_hi = x_offset, o_lo = out_offset, o_hi = out_offset;
  for (int d = 0; d < rank; d++) {
    if (region[d] < 0) return ctx->fail(TFHIP_EINVAL, "strided copy: negative extent");
    b.region[d] = region[d];
    b.x_stride[d] = x_strides[d];
    b.out_stride[d] = out_strides[d];
    n *= region[d];
    if (region[d] > 0) {
      const int64_t xs = x_strides[d] * (region[d] - 1), os = out_strides[d] * (region[d] - 1);
      if (xs < 0) x_lo += xs; else x_hi += xs;
      if (os < 0) o_lo += os; else o_hi += os;
    }
  }
  if (n == 0) return TFHIP_OK;
  if (x_lo < 0 || x_hi >= bx->numel || o_lo < 0 || o_hi >= bo->numel)
    return ctx->fail(TFHIP_EINVAL, "strided copy: the box leaves a buffer (source %lld..%lld of "
                                   "%lld, destination %lld..%lld of %lld)",
                     (long long)x_lo, (long long)x_hi, (long long)bx->numel, (long long)o_lo,
                     (long long)o_hi, (long long)bo->numel);
  if (bx->ptr == bo->ptr) return ctx->fail(TFHIP_EINVAL, "strided copy: in place is not supported");
  const dim3 grid(grid_for(ctx, n, 256)), block(256);
  // (indices of the elements in flight past the last one stay below 2^31 too)
  if (x_hi <= INDEX32 && o_hi <= INDEX32 && n <= INDEX32 - 4LL * 256 * grid.x) {
    Box32 c = {};
    c.x_offset = (int32_t)x_offset;
    c.out_offset = (int32_t)out_offset;
    int64_t extent[MAXBOX];
    for (int d = 0; d < rank; d++) {
      if (region[d] == 1) continue;
      // an outer dimension whose step is the whole of this one on both sides joins it
      const int l = c.rank - 1;
      if (l >= 0 && c.x_stride[l] == x_strides[d] * region[d] && c.out_stride[l] == out_strides[d] * region[d]) {
        extent[l] *= region[d];
        c.x_stride[l] = (int32_t)x_strides[d];
        c.out_stride[l] = (int32_t)out_strides[d];
        continue;
      }
      extent[c.rank] = region[d];
      c.x_stride[c.rank] = (int32_t)x_strides[d];
      c.out_stride[c.rank++] = (int32_t)out_strides[d];
    }
    // Runs: the innermost dimension side by side on both sides, or a mirrored row of small pixels.  (Below 8
    // elements, or 8 pixels, a row's last vector repeats too much of the one before.)
    const bool words = dtype_size(bx->dtype) == 4;
    auto inner = [&](int from_end, int64_t xs) {
      const int d = c.rank - from_end;
      return d >= 0 && c.x_stride[d] == xs && c.out_stride[d] == (xs < 0 ? -xs : xs) && extent[d] >= 8;
    };
    const int64_t pixel = c.rank > 0 && c.x_stride[c.rank - 1] == 1 && c.out_stride[c.rank - 1] == 1 ? extent[c.rank - 1] : 0;
    int mirror = -1, drop = 1;
    if (words && inner(1, 1)) mirror = 0;
    else if (words && inner(1, -1)) mirror = 1;
    else if (words && (pixel == 2 || pixel == 3) && inner(2, -pixel)) mirror = (int)pixel, drop = 2;
    for (int d = 0; d < c.rank; d++) c.region[d] = Divisor(extent[d]);
    if (mirror >= 0) {
      const int64_t len = extent[c.rank - drop] * (mirror > 1 ? mirror : 1), groups = ceil_div(len, 4);
      c.rank -= drop;
      int64_t lanes = groups;
      for (int d = 0; d < c.rank; d++) lanes *= extent[d];
      auto kernel = mirror == 0   ? copy_runs_kernel<0>
                    : mirror == 1 ? copy_runs_kernel<1>
                    : mirror == 2 ? copy_runs_kernel<2>
                                  : copy_runs_kernel<3>;
      tfhip::launch(ctx, kernel, dim3((unsigned)ceil_div(lanes, 256)), block, 0, (const int32_t*)bx->ptr,
                    (int32_t*)bo->ptr, (uint32_t)lanes, c, Divisor(groups), (int)len);
      TFHIP_LAUNCH_CHECK(ctx);
      return TFHIP_OK;
    }
    const dim3 grid4(grid_for(ctx, ceil_div(n, 4), 256));
    if (words)
      tfhip::launch(ctx, strided_copy32_kernel<int32_t>, grid4, block, 0, (const int32_t*)bx->ptr,
                    (int32_t*)bo->ptr, (uint32_t)n, c);
    else
      tfhip::launch(ctx, strided_copy32_kernel<uint8_t>, grid4, block, 0, (const uint8_t*)bx->ptr,
                    (uint8_t*)bo->ptr, (uint32_t)n, c);
    TFHIP_LAUNCH_CHECK(ctx);
    return TFHIP_OK;
  }
  if (dtype_size(bx->dtype) == 4)
    tfhip::launch(ctx, strided_copy_kernel<int32_t>, grid, block, 0,
                       (const int32_t*)bx->ptr, (int32_t*)bo->ptr, n, b);
  else
    tfhip::launch(ctx, strided_copy_kernel<uint8_t>, grid, block, 0,
                       (const uint8_t*)bx->ptr, (uint8_t*)bo->ptr, n, b);
  TFHIP_LAUNCH_CHECK(ctx);
  return TFHIP_OK;
}

extern "C" int tfhip_logical_not(tfhip_ctx* ctx, int64_t x, int64_t out) {
  if (!ctx) return TFHIP_EINVAL;
  TFHIP_GET(ctx, bx, x);
  TFHIP_GET(ctx, bo, out);
  if (bx->dtype != TFHIP_BOOL || bo->dtype != TFHIP_BOOL || bx->numel != bo->numel)
    return ctx->fail(TFHIP_EINVAL, "logicalNot: operand and result must be bool of one size");
  if (bx->numel == 0) return TFHIP_OK;
  tfhip::launch(ctx, logical_not_kernel, dim3(grid_for(ctx, bx->numel, 256)), dim3(256), 0, (const uint8_t*)bx->ptr, (uint8_t*)bo->ptr, bx->numel);
  TFHIP_LAUNCH_CHECK(ctx);
  return TFHIP_OK;
}

extern "C" int tfhip_batchnorm(tfhip_ctx* ctx, int64_t x, int64_t mean, int64_t variance,
                               int64_t offset, int64_t scale, float epsilon, int64_t out) {
  if (!ctx) return TFHIP_EINVAL;
  TFHIP_GET(ctx, bx, x);
  TFHIP_GET(ctx, bm, mean);
  TFHIP_GET(ctx, bv, variance);
  TFHIP_GET(ctx, bo, out);
  tfhip::Buf *boff = nullptr, *bs = nullptr;
  if (offset >= 0 && !(boff = ctx->find(offset))) return TFHIP_ENOENT;
  if (scale >= 0 && !(bs = ctx->find(scale))) return TFHIP_ENOENT;
  if (bo->dtype != TFHIP_FLOAT32 || bo->numel != bx->numel)
    return ctx->fail(TFHIP_EINVAL, "batchNorm: result must be float32 of the size of x");
  if (bx->numel == 0) return TFHIP_OK;
  if (bm->numel == 0 || bv->numel == 0 || (boff && boff->numel == 0) || (bs && bs->numel == 0))
    return ctx->fail(TFHIP_EINVAL, "batchNorm: empty statistics");
  Temp tx(ctx), tm(ctx), tv(ctx), to(ctx), ts(ctx);
  const float *xf, *mf, *vf, *of = nullptr, *sf = nullptr;
  int rc;
  if ((rc = as_f32(ctx, bx, &tx, &xf)) || (rc = as_f32(ctx, bm, &tm, &mf)) ||
      (rc = as_f32(ctx, bv, &tv, &vf)))
    return rc;
  if (boff && (rc = as_f32(ctx, boff, &to, &of))) return rc;
  if (bs && (rc = as_f32(ctx, bs, &ts, &sf))) return rc;
  const int64_t c = bm->numel, n = bx->numel;
  auto al = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  if (c % 4 == 0 && n % c == 0 && n / 4 <= INDEX32 / 2 && bv->numel == c && (!boff || boff->numel == c) &&
      (!bs || bs->numel == c) && al(xf) && al(mf) && al(vf) && al(of) && al(sf) && al(bo->ptr)) {
    tfhip::launch(ctx, batchnorm_channels_kernel, dim3(grid_for(ctx, n / 4, 256)), dim3(256), 0,
                  (const bn_f32x4*)xf, (const bn_f32x4*)mf, (const bn_f32x4*)vf, (const bn_f32x4*)of,
                  (const bn_f32x4*)sf, epsilon, (bn_f32x4*)bo->ptr, (uint32_t)(n / 4), Divisor(c / 4));
    TFHIP_LAUNCH_CHECK(ctx);
    return TFHIP_OK;
  }
  tfhip::launch(ctx, batchnorm_kernel, dim3(grid_for(ctx, bx->numel, 256)), dim3(256), 0, xf, mf, bm->numel, vf, bv->numel, of, boff ? boff->numel : 1, sf,
                     bs ? bs->numel : 1, epsilon, (float*)bo->ptr, bx->numel);
  TFHIP_LAUNCH_CHECK(ctx);
  return TFHIP_OK;
}

extern "C" int tfhip_resize_bilinear(tfhip_ctx* ctx, int64_t x, int64_t out, int batch, int in_h,
                                     int in_w, int channels, int out_h, int out_w,
                                     int align_corners) {
  if (!ctx) return TFHIP_EINVAL;
  TFHIP_GET(ctx, bx, x);
  TFHIP_GET(ctx, bo, out);
  if (batch < 0 || in_h < 0 || in_w < 0 || channels < 0 || out_h < 0 || out_w < 0)
    return ctx->fail(TFHIP_EINVAL, "resizeBilinear: bad geometry");
  if (bx->numel != (int64_t)batch * in_h * in_w * channels ||
      bo->numel != (int64_t)batch * out_h * out_w * channels || bo->dtype != TFHIP_FLOAT32)
    return ctx->fail(TFHIP_EINVAL, "resizeBilinear: buffers do not match the shapes given");
  if (bo->numel == 0) return TFHIP_OK;
  if (in_h == 0 || in_w == 0) return ctx->fail(TFHIP_EINVAL, "resizeBilinear: empty input image");
  Temp tx(ctx);
  const float* xf;
  int rc;
  if ((rc = as_f32(ctx, bx, &tx, &xf))) return rc;
  // effective sizes and ratios (backend_cpu.ts:2885-2898)
  const double eh_in = (align_corners && out_h > 1) ? in_h - 1 : in_h;
  const double ew_in = (align_corners && out_w > 1) ? in_w - 1 : in_w;
  const double eh_out = (align_corners && out_h > 1) ? out_h - 1 : out_h;
  const double ew_out = (align_corners && out_w > 1) ? out_w - 1 : out_w;
  if (const int vec = resize_width(bx, xf, bo, channels)) {
    const ResizePlan p = resize_plan(bo->numel, vec, channels, in_h, in_w, out_h, out_w, eh_in / eh_out, ew_in / ew_out);
    const dim3 grid((unsigned)ceil_div(p.n, 256)), block(256);
    typedef Channels<4>::T Four;
    if (vec == 4) tfhip::launch(ctx, resize_bilinear32_kernel<4>, grid, block, 0, (const Four*)xf, (Four*)bo->ptr, p);
    else tfhip::launch(ctx, resize_bilinear32_kernel<1>, grid, block, 0, xf, (float*)bo->ptr, p);
    TFHIP_LAUNCH_CHECK(ctx);
    return TFHIP_OK;
  }
  tfhip::launch(ctx, resize_bilinear_kernel, dim3(grid_for(ctx, bo->numel, 256)), dim3(256), 0, xf, (float*)bo->ptr, batch, in_h, in_w, channels, out_h, out_w,
                     eh_in / eh_out, ew_in / ew_out);
  TFHIP_LAUNCH_CHECK(ctx);
  return TFHIP_OK;
}

extern "C" int tfhip_one_hot(tfhip_ctx* ctx, int64_t indices, int64_t out, int depth,
                             float on_value, float off_value) {
  if (!ctx) return TFHIP_EINVAL;
  TFHIP_GET(ctx, bi, indices);
  TFHIP_GET(ctx, bo, out);
  if (bi->dtype != TFHIP_INT32) return ctx->fail(TFHIP_EINVAL, "oneHot: indices must be int32");
  if (depth < 0 || bo->numel != bi->numel * depth ||
      (bo->dtype != TFHIP_INT32 && bo->dtype != TFHIP_FLOAT32))
    return ctx->fail(TFHIP_EINVAL, "oneHot: result must hold indices x depth int32 or float32 values");
  if (bo->numel == 0) return TFHIP_OK;
  const dim3 grid(grid_for(ctx, bo->numel, 256)), block(256);
  if (bo->dtype == TFHIP_INT32)
    tfhip::launch(ctx, one_hot_kernel<int32_t>, grid, block, 0,
                       (const int32_t*)bi->ptr, (int32_t*)bo->ptr, bi->numel, depth,
                       (int32_t)on_value, (int32_t)off_value);
  else
    tfhip::launch(ctx, one_hot_kernel<float>, grid, block, 0,
                       (const int32_t*)bi->ptr, (float*)bo->ptr, bi->numel, depth, on_value,
                       off_value);
  TFHIP_LAUNCH_CHECK(ctx);
  return TFHIP_OK;
}

extern "C" int tfhip_resize_nearest(tfhip_ctx* ctx, int64_t x, int64_t out, int batch, int in_h,
                                    int in_w, int channels, int out_h, int out_w,
                                    int align_corners) {
  if (!ctx) return TFHIP_EINVAL;
  TFHIP_GET(ctx, bx, x);
  TFHIP_GET(ctx, bo, out);
  if (batch < 0 || in_h < 0 || in_w < 0 || channels < 0 || out_h < 0 || out_w < 0)
    return ctx->fail(TFHIP_EINVAL, "resizeNearestNeighbor: bad geometry");
  if (bx->numel != (int64_t)batch * in_h * in_w * channels ||
      bo->numel != (int64_t)batch * out_h * out_w * channels || bo->dtype != TFHIP_FLOAT32)
    return ctx->fail(TFHIP_EINVAL, "resizeNearestNeighbor: buffers do not match the shapes given");
  if (bo->numel == 0) return TFHIP_OK;
  if (in_h == 0 || in_w == 0) return ctx->fail(TFHIP_EINVAL, "resizeNearestNeighbor: empty input image");
  Temp tx(ctx);
  const float* xf;
  int rc;
  if ((rc = as_f32(ctx, bx, &tx, &xf))) return rc;
  // effective sizes and ratios (backend_cpu.ts:3025-3038)
  const double eh_in = (align_corners && out_h > 1) ? in_h - 1 : in_h;
  const double ew_in = (align_corners && out_w > 1) ? in_w - 1 : in_w;
  const double eh_out = (align_corners && out_h > 1) ? out_h - 1 : out_h;
  const double ew_out = (align_corners && out_w > 1) ? out_w - 1 : out_w;
  if (const int vec = resize_width(bx, xf, bo, channels)) {
    const ResizePlan p = resize_plan(bo->numel, vec, channels, in_h, in_w, out_h, out_w, eh_in / eh_out, ew_in / ew_out);
    const dim3 grid((unsigned)ceil_div(p.n, 256)), block(256);
    typedef Channels<4>::T Four;
    if (vec == 4) tfhip::launch(ctx, resize_nearest32_kernel<4>, grid, block, 0, (const Four*)xf, (Four*)bo->ptr, p, align_corners);
    else tfhip::launch(ctx, resize_nearest32_kernel<1>, grid, block, 0, xf, (float*)bo->ptr, p, align_corners);
    TFHIP_LAUNCH_CHECK(ctx);
    return TFHIP_OK;
  }
  tfhip::launch(ctx, resize_nearest_kernel, dim3(grid_for(ctx, bo->numel, 256)), dim3(256), 0, xf, (float*)bo->ptr, batch, in_h, in_w, channels, out_h, out_w,
                     eh_in / eh_out, ew_in / ew_out, align_corners ? 1 : 0);
  TFHIP_LAUNCH_CHECK(ctx);
  return TFHIP_OK;
}

extern "C" int tfhip_select(tfhip_ctx* ctx, int64_t condition, int64_t a, int64_t b, int64_t out,
                            int64_t inner) {
  if (!ctx) return TFHIP_EINVAL;
  TFHIP_GET(ctx, bc, condition);
  TFHIP_GET(ctx, ba, a);
  TFHIP_GET(ctx, bb, b);
  TFHIP_GET(ctx, bo, out);
  if (bc->dtype != TFHIP_BOOL) return ctx->fail(TFHIP_EINVAL, "select: condition must be bool");
  if (ba->dtype == TFHIP_UINT8Q || ba->dtype != bb->dtype || ba->dtype != bo->dtype)
    return ctx->fail(TFHIP_EINVAL, "select: a, b and the result must share one storage dtype");
  if (inner < 1 || ba->numel != bb->numel || ba->numel != bo->numel ||
      bc->numel * inner != ba->numel)
    return ctx->fail(TFHIP_EINVAL, "select: sizes do not match (condition %lld x %lld, a %lld, b %lld)",
                     (long long)bc->numel, (long long)inner, (long long)ba->numel,
                     (long long)bb->numel);
  if (bo->numel == 0) return TFHIP_OK;
  const dim3 grid(grid_for(ctx, bo->numel, 256)), block(256);
  const uint8_t* c = static_cast<const uint8_t*>(bc->ptr);
  if (dtype_size(ba->dtype) == 4)
    tfhip::launch(ctx, select_kernel<int32_t>, grid, block, 0, c,
                       (const int32_t*)ba->ptr, (const int32_t*)bb->ptr, (int32_t*)bo->ptr,
                       bo->numel, inner);
  else
    tfhip::launch(ctx, select_kernel<uint8_t>, grid, block, 0, c,
                       (const uint8_t*)ba->ptr, (const uint8_t*)bb->ptr, (uint8_t*)bo->ptr,
                       bo->numel, inner);
  TFHIP_LAUNCH_CHECK(ctx);
  return TFHIP_OK;
}
