// Index-driven data movement and the resampling kernels around it: gatherND, scatterND /
// sparseToDense, resizeBilinearBackprop, resizeNearestNeighborBackprop, cropAndResize.
// Replaces backend_cpu.ts:2938-3013, 3070-3165, 3622-3757, 3759-3836, 3842-3889 of the
// reference.  Every result element is the sum of its contributions in the order the reference's
// loops visit them, so sums round the same way, with one exception: sums in double that are rounded once
// (unsortedSegmentSum) are taken in parts where a row has very many entries
// (scatter_groups_kernel), in an order that the indices alone decide.  Nothing depends on scheduling (no
// atomics on data).
#include <algorithm>
#include <climits>
#include <type_traits>

#include "tfhip_internal.h"

// The reference rounds every product before it adds it (JavaScript has no fused multiply-add);
// a contracted a * b + c keeps more bits and now and then lands on the neighbouring float32 or
// on the other side of an integer coordinate.
#pragma clang fp contract(off)

namespace tfhip {

constexpr int MAX_SLICE_RANK = 8;
struct SliceStrides {
  int rank;
  int64_t stride[MAX_SLICE_RANK];
};

static unsigned blocks_for(tfhip_ctx* ctx, int64_t items) {
  const int64_t blocks = (items + 255) / 256;
  const int64_t cap = (int64_t)ctx->num_cus * 16;
  return (unsigned)(blocks < 1 ? 1 : blocks > cap ? cap : blocks);
}

__global__ void set_int_kernel(int* p, int v) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *p = v;
}

// flat[i] = sum_j indices[i, j] * stride[j] (in units of slices); the smallest i whose flat
// index falls outside [0, rows) lands in *first_bad.
__global__ void flatten_indices_kernel(const int32_t* indices, int64_t* flat, int64_t n,
                                       SliceStrides s, int64_t rows, int* first_bad) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    int64_t f = 0;
    for (int j = 0; j < s.rank; j++) f += (int64_t)indices[i * s.rank + j] * s.stride[j];
    flat[i] = f;
    if (f < 0 || f >= rows) atomicMin(first_bad, (int)(i < INT_MAX ? i : INT_MAX - 1));
  }
}

template <typename T>
__global__ void gather_rows_kernel(const T* x, const int64_t* flat, T* out, int64_t n_slices,
                                   int64_t slice) {
  const int64_t total = n_slices * slice;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += stride) {
    const int64_t i = g / slice, k = g - i * slice;
    out[g] = x[flat[i] * slice + k];
  }
}

// The same copy in 16-byte pieces, for slices that are a whole number of them.
__global__ void gather_rows_vec_kernel(const uint4* x, const int64_t* flat, uint4* out, int64_t n_slices,
                                       int64_t slice16) {
  const int64_t total = n_slices * slice16;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += stride) {
    const int64_t i = g / slice16, k = g - i * slice16;
    out[g] = x[flat[i] * slice16 + k];
  }
}

// One lane per result element (row, k): starts from the default value and walks the updates
// in ascending order, adding (scatterND) or overwriting (sparseToDense: the last one wins)
// whenever an update addresses its row, which is the order backend_cpu.ts:3858-3886 applies
// them in.  Acc = T rounds every sum to the element type as a typed array does; Acc = double
// rounds once at the end, as the masked sums of unsortedSegmentSum do.
template <typename T, typename Acc, typename I>
__global__ __launch_bounds__(256) void scatter_rows_kernel(const I* flat, const T* updates, T* out,
                                                           int64_t rows, int64_t slice, int64_t n_updates,
                                                           T start, int sum_dupes, int scalar_update) {
  // the index list passes through LDS 256 entries at a time: every lane of the workgroup walks
  // the same entries, which LDS serves as broadcasts
  __shared__ int chunk[256];  // row of each update, -2 for none (rows fit an int: checked by the host)
  const int64_t total = rows * slice;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  // all lanes of a workgroup make the same number of trips, so the barriers below are uniform
  for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < total; base += stride) {
    const int64_t g = base + threadIdx.x;
    const bool live = g < total;
    const int row = live ? (int)(g / slice) : -1;
    const int64_t k = live ? g - (int64_t)row * slice : 0;
    Acc acc = start;
    for (int64_t i0 = 0; i0 < n_updates; i0 += 256) {
      __syncthreads();
      const int64_t f = i0 + threadIdx.x < n_updates ? flat[i0 + threadIdx.x] : -2;
      chunk[threadIdx.x] = f >= 0 && f < rows ? (int)f : -2;
      __syncthreads();
      // eight entries per trip, read together so that their LDS latencies overlap
      for (int j0 = 0; j0 < 256; j0 += 8) {
        int c[8];
#pragma unroll
        for (int e = 0; e < 8; e++) c[e] = chunk[j0 + e];
#pragma unroll
        for (int e = 0; e < 8; e++) {
          if (c[e] != row) continue;
          const T u = updates[scalar_update ? 0 : (i0 + j0 + e) * slice + k];
          acc = sum_dupes ? (Acc)(acc + u) : (Acc)u;
        }
      }
    }
    if (live) out[g] = (T)acc;
  }
}

// The same for slices of 32 elements and more (an embedding's gradient).  The kernel above walks
// the whole index list for every 256 result elements, which is what it is bound by: 10240 updates
// of 128 into 20000 rows took 1980 us; 25.5 here.  A workgroup of 16 or 4 wavefronts owns the rows f with
// f % groups = its number (so that the frequent rows of a text, which have neighbouring numbers,
// go to different workgroups) and 64 columns for each of CW wavefronts side by side: it walks the
// list once, 4096 entries at a time, and packs the entries of its rows, in order, into LDS, counting
// them per row.  A set of CW wavefronts then takes a row that has any, finds its entries by ballot
// and adds them in ascending order, up to 64 updates in flight.  What bounds it is the most frequent
// row, a chain of hundreds of additions: sums that are rounded once at the end (Acc = double) of a
// row with more than HOT entries in the pass are cut over the sets, 64 list entries in turn each,
// and their parts added in the order of the sets (one set for the whole chain, four wavefronts: 64 us).
// The sums lie in LDS between passes; every other one is taken in the order of the list, as above.
constexpr int SCATTER_PASS = 4096;
template <typename T, typename Acc, int CW, int THREADS, typename I>
__global__ __launch_bounds__(THREADS) void scatter_groups_kernel(
    const I* __restrict__ flat, const T* __restrict__ updates, T* __restrict__ out, int rows, int64_t slice,
    int64_t n_updates, T start, int sum_dupes, int scalar_update, int group_shift, int local_rows) {
  constexpr int WAVES = THREADS / 64, PER = SCATTER_PASS / THREADS, CB = 64 * CW, SETS = WAVES / CW;
  static_assert(PER * WAVES == 64, "the counts of a pass are one wavefront's prefix sum");
  constexpr bool CUT = !std::is_same<T, Acc>::value && SETS > 1;
  constexpr int HOT = 64;
  extern __shared__ __attribute__((aligned(16))) char scatter_lds[];
  Acc* sums = reinterpret_cast<Acc*>(scatter_lds);               // [local_rows][CB]
  int* counts = reinterpret_cast<int*>(sums + local_rows * CB);  // entries of the pass per row
  __shared__ unsigned list[SCATTER_PASS];                        // local row << 12 | entry of the pass
  __shared__ int first[65];                                      // where a wavefront's entries of a load begin
  __shared__ Acc parts[CUT ? SETS * CB : 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int groups = 1 << group_shift, mine = (int)(blockIdx.z * gridDim.x + blockIdx.x);
  const int set = wave / CW, own = (wave % CW) * 64 + lane;      // column within the block
  const int64_t col = (int64_t)blockIdx.y * CB + own;
  const bool stored = col < slice;
  const int64_t read_col = stored ? col : 0;                     // (a column past the slice: summed, not stored)
  for (int i = tid; i < local_rows * CB; i += THREADS) sums[i] = (Acc)start;
  for (int64_t i0 = 0; i0 < n_updates; i0 += SCATTER_PASS) {
    for (int i = tid; i < local_rows; i += THREADS) counts[i] = 0;
    I f[PER];
#pragma unroll
    for (int u = 0; u < PER; u++) {
      const int64_t i = i0 + u * THREADS + tid;
      f[u] = i < n_updates ? flat[i] : -1;
    }
    unsigned long long hit[PER];
#pragma unroll
    for (int u = 0; u < PER; u++) {
      const bool in = f[u] >= 0 && f[u] < rows && ((int)f[u] & (groups - 1)) == mine;
      hit[u] = __ballot(in);
      if (lane == 0) first[u * WAVES + wave] = __popcll(hit[u]);
    }
    __syncthreads();
    if (wave == 0) {  // 64 counts into their prefix sums
      int n = first[lane];
      const int count = n;
      for (int off = 1; off < 64; off <<= 1) {
        const int o = __shfl_up(n, off, 64);
        if (lane >= off) n += o;
      }
      first[lane] = n - count;
      if (lane == 63) first[64] = n;
    }
    __syncthreads();
    const int total = __builtin_amdgcn_readfirstlane(first[64]);
#pragma unroll
    for (int u = 0; u < PER; u++)
      if (hit[u] >> lane & 1) {
        const int r = (int)f[u] >> group_shift;
        list[first[u * WAVES + wave] + __popcll(hit[u] & ((1ull << lane) - 1))] =
            (unsigned)r << 12 | (unsigned)(u * THREADS + tid);
        atomicAdd(&counts[r], 1);
      }
    __syncthreads();
    const T* pass_updates = updates + (scalar_update ? 0 : i0 * slice);
    const int64_t step = scalar_update ? 0 : slice;
    const int64_t at_col = scalar_update ? 0 : read_col;
    // the entries of row r among list[c0 .. c0 + 64), added to acc in ascending order
    auto add_entries = [&](int r, int c0, Acc& acc) {
      const unsigned e = c0 + lane < total ? list[c0 + lane] : ~0u;
      unsigned long long left = __ballot((int)(e >> 12) == r);
      const int found = (int)__popcll(left);
      // up to U updates in flight.  (No branches around the loads, or each would be waited
      // for: past the last entry the one before is read again.)
      auto take = [&](auto most) {
        constexpr int U = decltype(most)::value;
        T x[U];
        const int n = min(U, (int)__popcll(left));
        int at = 0;
#pragma unroll
        for (int u = 0; u < U; u++) {
          at = left ? __builtin_ctzll(left) : at;
          left &= left - 1;
          const int entry = __builtin_amdgcn_readlane((int)e, at) & (SCATTER_PASS - 1);
          x[u] = (pass_updates + entry * step)[at_col];
        }
#pragma unroll
        for (int u = 0; u < U; u++)
          if (u < n) acc = sum_dupes ? (Acc)(acc + x[u]) : (Acc)x[u];
      };
      while (left) {
        const int n = __popcll(left);
        if (n > 16) take(std::integral_constant<int, 64>());
        else if (n > 2) take(std::integral_constant<int, 16>());
        else take(std::integral_constant<int, 2>());
      }
      return found;
    };
    for (int r0 = 0; r0 < local_rows && total > 0; r0 += 64) {
      const int n = r0 + lane < local_rows ? counts[r0 + lane] : 0;
      // (the same masks in every wavefront)
      unsigned long long hot = CUT && sum_dupes ? __ballot(n > HOT) : 0ull;
      unsigned long long mine_left = __ballot(n > 0) & ~hot & (~0ull / ((1ull << SETS) - 1)) << set;
      for (; mine_left; mine_left &= mine_left - 1) {
        const int at = __builtin_ctzll(mine_left), r = r0 + at;
        int due = __builtin_amdgcn_readlane(n, at);
        Acc acc = sums[r * CB + own];
        for (int c0 = 0; due > 0; c0 += 64) due -= add_entries(r, c0, acc);
        sums[r * CB + own] = acc;
      }
      if constexpr (CUT) {
        for (; hot; hot &= hot - 1) {
          const int r = r0 + __builtin_ctzll(hot);
          Acc acc = (Acc)0;
          for (int c0 = set * 64; c0 < total; c0 += 64 * SETS) add_entries(r, c0, acc);
          parts[set * CB + own] = acc;
          __syncthreads();
          if (set == 0) {
            Acc all = sums[r * CB + own];
            for (int s = 0; s < SETS; s++) all += parts[s * CB + own];
            sums[r * CB + own] = all;
          }
          __syncthreads();
        }
      }
    }
    __syncthreads();
  }
  __syncthreads();
  for (int r = set; r < local_rows; r += SETS) {
    const int64_t row = mine + (int64_t)r * groups;
    if (row >= rows) break;
    if (stored) out[row * slice + col] = (T)sums[r * CB + own];
  }
}

// log2 of the groups: enough that a group's sums fit, and `per_cu` workgroups per CU where there are
// rows for them.
static constexpr int scatter_group_shift(int64_t rows, int64_t col_blocks, int most_local, int cus, int per_cu = 4) {
  int shift = 0;
  while ((rows + ((int64_t)1 << shift) - 1) >> shift > most_local ||
         (((int64_t)1 << shift) * col_blocks < per_cu * cus && ((int64_t)2 << shift) <= rows))
    shift++;
  return shift;
}
// A launch counts its lanes along a dimension in 32 bits: 2^21 groups of 1024 side by side, four
// times.  (168 million rows of 129 columns in double, 87 GB, are the first that need more.)
constexpr int SCATTER_MOST_SHIFT = 23, SCATTER_SHIFT_X = 21;
static_assert(scatter_group_shift(20ll << 23, 1, 20, 256) == SCATTER_MOST_SHIFT &&
              scatter_group_shift((20ll << 23) + 1, 1, 20, 256) > SCATTER_MOST_SHIFT, "");
static_assert(scatter_group_shift(20000, 1, 80, 256) == 10 && scatter_group_shift(1, 1, 80, 256) == 0, "");

// False: too many rows for this kernel.
template <typename T, typename Acc, int CW, typename I>
static bool launch_scatter_groups(tfhip_ctx* ctx, const I* flat, const T* updates, T* out, int rows,
                                  int64_t slice, int64_t n_updates, T start, int sum_dupes, int scalar_update) {
  constexpr int CB = 64 * CW, MOST_LOCAL = (40 << 10) / (CB * (int)sizeof(Acc));  // 40 KB of sums
  const int64_t col_blocks = ceil_div(slice, CB);
  // 16 wavefronts where all workgroups are in the machine at once (two a CU) or nearly: one pass over the
  // list takes as long as its longest chain.  With more of them, what counts is how often the list is walked,
  // and four wavefronts walk it in fewer steps: 100000 rows of 300, 50000 updates 790 us against 1366 (and
  // 20000 rows of 128, 10240 updates 25.5 with sixteen, 50 with four).  A short list has no long chains.
  int shift = scatter_group_shift(rows, col_blocks, MOST_LOCAL, ctx->num_cus, 2);
  const bool wide = ((int64_t)1 << shift) * col_blocks <= 4 * ctx->num_cus && n_updates > 1024;
  if (!wide) shift = scatter_group_shift(rows, col_blocks, MOST_LOCAL, ctx->num_cus);
  if (shift > SCATTER_MOST_SHIFT) return false;
  const int local_rows = (int)ceil_div(rows, (int64_t)1 << shift), across = std::min(shift, SCATTER_SHIFT_X);
  tfhip::launch(ctx, wide ? scatter_groups_kernel<T, Acc, CW, 1024, I> : scatter_groups_kernel<T, Acc, CW, 256, I>,
                dim3(1u << across, (unsigned)col_blocks, 1u << (shift - across)), dim3(wide ? 1024 : 256),
                (size_t)local_rows * (CB * sizeof(Acc) + sizeof(int)), flat, updates, out, rows, slice, n_updates, start,
                sum_dupes, scalar_update, shift, local_rows);
  return true;
}
template <typename T, typename Acc, typename I>
static void launch_scatter(tfhip_ctx* ctx, const I* flat, const T* updates, T* out, int64_t rows,
                           int64_t slice, int64_t n_updates, T start, int sum_dupes, int scalar_update) {
  // (half a wavefront of columns, and column blocks that a grid's second dimension holds)
  if (slice >= 32 && n_updates > 0 && slice <= 65535 * 256) {
    auto launch = slice <= 64    ? launch_scatter_groups<T, Acc, 1, I>
                  : slice <= 128 ? launch_scatter_groups<T, Acc, 2, I>
                                 : launch_scatter_groups<T, Acc, 4, I>;
    if (launch(ctx, flat, updates, out, (int)rows, slice, n_updates, start, sum_dupes, scalar_update)) return;
  }
  tfhip::launch(ctx, (scatter_rows_kernel<T, Acc, I>), dim3(blocks_for(ctx, rows * slice)), dim3(256), 0, flat,
                updates, out, rows, slice, n_updates, start, sum_dupes, scalar_update);
}

// Source rows / columns of a resized pixel as the reference computes them, in double.
struct Lerp {
  int lo, hi;
  double w;  // weight of hi; 1 - w goes to lo
};
__device__ inline Lerp lerp_at(int r, double scale, int in_size) {
  const double f = r * scale;
  Lerp l;
  l.lo = (int)floor(f);
  l.hi = min((int)ceil(f), in_size - 1);
  l.w = f - l.lo;
  return l;
}
// The resized rows whose source rows can touch input row y: r * scale within (y - 1, y + 1),
// widened by one either side against rounding of the division.
__device__ inline void touching(int y, double scale, int out_size, int* lo, int* hi) {
  if (!(scale > 0.0)) {
    *lo = 0;
    *hi = out_size - 1;
    return;
  }
  const double a = floor((y - 1) / scale) - 1.0, b = ceil((y + 1) / scale) + 1.0;
  *lo = a < 0.0 ? 0 : (a > out_size - 1 ? out_size - 1 : (int)a);
  *hi = b > out_size - 1 ? out_size - 1 : (b < 0.0 ? 0 : (int)b);
}

// dx[b, y, x, d]: every dy pixel (r, c) spreads over its four source pixels with the bilinear
// weights; this lane collects what lands on (y, x), in ascending (r, c) and, within one
// pixel, in the order top-left, top-right, bottom-left, bottom-right (backend_cpu.ts:2967-3009).
// The running sum is a float32 that takes one double-precision add per contribution, like a
// Float32Array element.
__global__ void resize_bilinear_backprop_kernel(const float* dy, float* dx, int batch, int x_h,
                                                int x_w, int ch, int y_h, int y_w,
                                                double scale_h, double scale_w) {
  const int64_t n = (int64_t)batch * x_h * x_w * ch;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const int d = (int)(i % ch);
    int64_t t = i / ch;
    const int x = (int)(t % x_w);
    t /= x_w;
    const int y = (int)(t % x_h);
    const int b = (int)(t / x_h);
    int r_lo, r_hi, c_lo, c_hi;
    touching(y, scale_h, y_h, &r_lo, &r_hi);
    touching(x, scale_w, y_w, &c_lo, &c_hi);
    float acc = 0.f;
    for (int r = r_lo; r <= r_hi; r++) {
      const Lerp lr = lerp_at(r, scale_h, x_h);
      const bool top = lr.lo == y, bottom = lr.hi == y;
      if (!top && !bottom) continue;
      for (int c = c_lo; c <= c_hi; c++) {
        const Lerp lc = lerp_at(c, scale_w, x_w);
        const bool left = lc.lo == x, right = lc.hi == x;
        if (!left && !right) continue;
        const double g = dy[(((int64_t)b * y_h + r) * y_w + c) * ch + d];
        if (top && left) acc = (float)((double)acc + g * ((1.0 - lr.w) * (1.0 - lc.w)));
        if (top && right) acc = (float)((double)acc + g * ((1.0 - lr.w) * lc.w));
        if (bottom && left) acc = (float)((double)acc + g * (lr.w * (1.0 - lc.w)));
        if (bottom && right) acc = (float)((double)acc + g * (lr.w * lc.w));
      }
    }
    dx[i] = acc;
  }
}

// dx[b, y, x, d] = sum of the dy pixels whose nearest source pixel is (y, x), added in
// ascending (row, column) in double and rounded once (backend_cpu.ts:3107-3160).  The
// reference searches a window around y / scale; the rows that can qualify lie within
// `touching`, and rows outside its window never qualify, so both visit the same pixels.
__global__ void resize_nearest_backprop_kernel(const float* dy, float* dx, int batch, int x_h,
                                               int x_w, int ch, int y_h, int y_w, double scale_h,
                                               double scale_w, int align_corners) {
  const int64_t n = (int64_t)batch * x_h * x_w * ch;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const int d = (int)(i % ch);
    int64_t t = i / ch;
    const int x = (int)(t % x_w);
    t /= x_w;
    const int y = (int)(t % x_h);
    const int b = (int)(t / x_h);
    int r_lo, r_hi, c_lo, c_hi;
    touching(y, scale_h, y_h, &r_lo, &r_hi);
    touching(x, scale_w, y_w, &c_lo, &c_hi);
    double acc = 0.0;
    for (int r = r_lo; r <= r_hi; r++) {
      const double fr = r * scale_h;
      if (min(x_h - 1, (int)(align_corners ? floor(fr + 0.5) : floor(fr))) != y) continue;
      for (int c = c_lo; c <= c_hi; c++) {
        const double fc = c * scale_w;
        if (min(x_w - 1, (int)(align_corners ? floor(fc + 0.5) : floor(fc))) != x) continue;
        acc += dy[(((int64_t)b * y_h + r) * y_w + c) * ch + d];
      }
    }
    dx[i] = (float)acc;
  }
}

// One lane per element of the crops, channel fastest; coordinates in double from the
// float32 box corners, as backend_cpu.ts:3646-3753 computes them.  A box whose image index
// is outside the batch leaves zeros.
__global__ void crop_and_resize_kernel(const float* images, const float* boxes,
                                       const int32_t* box_index, float* out, int batch, int img_h,
                                       int img_w, int ch, int64_t n_boxes, int crop_h, int crop_w,
                                       int nearest, float extrapolation) {
  const int64_t n = n_boxes * crop_h * crop_w * ch;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const int c = (int)(i % ch);
    int64_t t = i / ch;
    const int x = (int)(t % crop_w);
    t /= crop_w;
    const int y = (int)(t % crop_h);
    const int64_t b = t / crop_h;
    const double y1 = boxes[b * 4], x1 = boxes[b * 4 + 1], y2 = boxes[b * 4 + 2],
                 x2 = boxes[b * 4 + 3];
    const int img = box_index[b];
    if (img < 0 || img >= batch) {
      out[i] = 0.f;
      continue;
    }
    const double scale_h = crop_h > 1 ? (y2 - y1) * (img_h - 1) / (crop_h - 1) : 0.0;
    const double scale_w = crop_w > 1 ? (x2 - x1) * (img_w - 1) / (crop_w - 1) : 0.0;
    const double fy = crop_h > 1 ? y1 * (img_h - 1) + y * scale_h : 0.5 * (y1 + y2) * (img_h - 1);
    const double fx = crop_w > 1 ? x1 * (img_w - 1) + x * scale_w : 0.5 * (x1 + x2) * (img_w - 1);
    // NaN coordinates fail both comparisons in the reference and read outside the image
    // there; here they extrapolate
    if (!(fy >= 0.0 && fy <= img_h - 1) || !(fx >= 0.0 && fx <= img_w - 1)) {
      out[i] = extrapolation;
      continue;
    }
    const float* im = images + (int64_t)img * img_h * img_w * ch + c;
    if (nearest) {
      const int cy = (int)floor(fy + 0.5), cx = (int)floor(fx + 0.5);
      out[i] = im[((int64_t)cy * img_w + cx) * ch];
    } else {
      const int top = (int)floor(fy), bottom = (int)ceil(fy);
      const int left = (int)floor(fx), right = (int)ceil(fx);
      const double wy = fy - top, wx = fx - left;
      const double tl = im[((int64_t)top * img_w + left) * ch], tr = im[((int64_t)top * img_w + right) * ch];
      const double bl = im[((int64_t)bottom * img_w + left) * ch],
                   br = im[((int64_t)bottom * img_w + right) * ch];
      const double up = tl + (tr - tl) * wx, down = bl + (br - bl) * wx;
      out[i] = (float)(up + (down - up) * wy);
    }
  }
}

// Flat slice indices of `indices` [n, slice_rank] into a tensor of `shape` whose first
// slice_rank dimensions are indexed; fails with the reference's message when one of them is
// out of range (backend_cpu.ts:3796-3799, 3870-3873).  Waits for the device.  as_they_are: the
// caller reads the indices themselves, only the shapes are looked at.
static int flatten_checked(tfhip_ctx* ctx, const char* op, const Buf* bi, const int32_t* shape,
                           int rank, int64_t n, int slice_rank, Temp* flat, int64_t* slice_out,
                           int64_t* rows_out, bool check = true, bool as_they_are = false) {
  if (check && ctx->capturing)
    return ctx->fail(TFHIP_EINVAL, "%s: checks its indices on the host, which a graph capture cannot do", op);
  if (rank < 0 || rank > MAX_SLICE_RANK || slice_rank < 0 || slice_rank > rank || n < 0)
    return ctx->fail(TFHIP_EINVAL, "%s: bad shape or index depth", op);
  if (bi->dtype != TFHIP_INT32) return ctx->fail(TFHIP_EINVAL, "%s: indices must be int32", op);
  if (bi->numel != n * slice_rank)
    return ctx->fail(TFHIP_EINVAL, "%s: indices do not hold %lld x %d values", op, (long long)n, slice_rank);
  SliceStrides s = {};
  s.rank = slice_rank;
  int64_t slice = 1, rows = 1;
  for (int d = rank - 1; d >= slice_rank; d--) slice *= shape[d];
  for (int d = slice_rank - 1; d >= 0; d--) {
    s.stride[d] = rows;
    rows *= shape[d];
  }
  *slice_out = slice;
  *rows_out = rows;
  if (n == 0 || as_they_are) return TFHIP_OK;
  Temp flag(ctx);
  if (!flat->get((size_t)n * sizeof(int64_t)) || !flag.get(sizeof(int))) return TFHIP_EDEVICE;
  int* bad = static_cast<int*>(flag.ptr);
  tfhip::launch(ctx, set_int_kernel, dim3(1), dim3(1), 0, bad, INT_MAX);
  tfhip::launch(ctx, flatten_indices_kernel, dim3(blocks_for(ctx, n)), dim3(256), 0,
                     (const int32_t*)bi->ptr, (int64_t*)flat->ptr, n, s, rows, bad);
  TFHIP_LAUNCH_CHECK(ctx);
  if (!check) return TFHIP_OK;
  int first_bad = INT_MAX;
  TFHIP_HIP(ctx, hipMemcpyAsync(&first_bad, bad, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
  TFHIP_HIP(ctx, hipStreamSynchronize(ctx->stream));
  if (first_bad == INT_MAX) return TFHIP_OK;
  int32_t idx[MAX_SLICE_RANK] = {0};
  TFHIP_HIP(ctx, hipMemcpy(idx, (const int32_t*)bi->ptr + (int64_t)first_bad * slice_rank,
                           sizeof(int32_t) * slice_rank, hipMemcpyDeviceToHost));
  char index_text[160] = "", shape_text[160] = "";
  for (int j = 0, at = 0; j < slice_rank && at < 140; j++)
    at += snprintf(index_text + at, sizeof index_text - at, j ? ",%d" : "%d", idx[j]);
  for (int j = 0, at = 0; j < rank && at < 140; j++)
    at += snprintf(shape_text + at, sizeof shape_text - at, j ? ",%d" : "%d", shape[j]);
  return ctx->fail(TFHIP_EINVAL, "Invalid indices: %s does not index into %s", index_text, shape_text);
}

static int resize_backprop_check(tfhip_ctx* ctx, const char* op, const Buf* bdy, const Buf* bdx,
                                 int batch, int x_h, int x_w, int ch, int y_h, int y_w) {
  if (batch < 0 || x_h < 0 || x_w < 0 || ch < 0 || y_h < 0 || y_w < 0)
    return ctx->fail(TFHIP_EINVAL, "%s: bad geometry", op);
  if (bdy->numel != (int64_t)batch * y_h * y_w * ch || bdx->numel != (int64_t)batch * x_h * x_w * ch ||
      bdy->dtype != TFHIP_FLOAT32 || bdx->dtype != TFHIP_FLOAT32)
    return ctx->fail(TFHIP_EINVAL, "%s: float32 buffers of the shapes given are required", op);
  return TFHIP_OK;
}

}  // namespace tfhip

using namespace tfhip;

extern "C" int tfhip_gather_nd(tfhip_ctx* ctx, int64_t x, int64_t indices, int64_t out,
                               const int32_t* x_shape, int rank, int64_t num_slices,
                               int slice_rank) {
  if (!ctx) return TFHIP_EINVAL;
  TFHIP_GET(ctx, bx, x);
  TFHIP_GET(ctx, bi, indices);
  TFHIP_GET(ctx, bo, out);
  if (rank > 0 && !x_shape) return ctx->fail(TFHIP_EINVAL, "gatherND: shape missing");
  Temp flat(ctx);
  int64_t slice = 0, rows = 0;
  int rc;
  if ((rc = flatten_checked(ctx, "gatherND", bi, x_shape, rank, num_slices, slice_rank, &flat, &slice, &rows)))
    return rc;
  if (bx->numel != rows * slice || bo->numel != num_slices * slice)
    return ctx->fail(TFHIP_EINVAL, "gatherND: buffer sizes do not match the shapes given");
  if (bx->dtype == TFHIP_UINT8Q || dtype_size(bx->dtype) != dtype_size(bo->dtype))
    return ctx->fail(TFHIP_EINVAL, "gatherND: input and output element sizes differ");
  if (bo->numel == 0) return TFHIP_OK;
  const dim3 grid(blocks_for(ctx, bo->numel)), block(256);
  const int64_t slice_bytes = slice * (int64_t)dtype_size(bx->dtype);
  if (slice_bytes % 16 == 0 && reinterpret_cast<uintptr_t>(bx->ptr) % 16 == 0 &&
      reinterpret_cast<uintptr_t>(bo->ptr) % 16 == 0)
    tfhip::launch(ctx, gather_rows_vec_kernel, dim3(blocks_for(ctx, num_slices * (slice_bytes / 16))), block, 0, (const uint4*)bx->ptr, (const int64_t*)flat.ptr, (uint4*)bo->ptr, num_slices,
                       slice_bytes / 16);
  else if (dtype_size(bx->dtype) == 4)
    tfhip::launch(ctx, gather_rows_kernel<int32_t>, grid, block, 0, (const int32_t*)bx->ptr,
                       (const int64_t*)flat.ptr, (int32_t*)bo->ptr, num_slices, slice);
  else
    tfhip::launch(ctx, gather_rows_kernel<uint8_t>, grid, block, 0, (const uint8_t*)bx->ptr,
                       (const int64_t*)flat.ptr, (uint8_t*)bo->ptr, num_slices, slice);
  TFHIP_LAUNCH_CHECK(ctx);
  return TFHIP_OK;
}

extern "C" int tfhip_scatter_nd(tfhip_ctx* ctx, int64_t indices, int64_t updates, int64_t out,
                                const int32_t* out_shape, int rank, int64_t num_updates,
                                int slice_rank, double default_value, int flags) {
  if (!ctx) return TFHIP_EINVAL;
  TFHIP_GET(ctx, bi, indices);
  TFHIP_GET(ctx, bu, updates);
  TFHIP_GET(ctx, bo, out);
  if (rank > 0 && !out_shape) return ctx->fail(TFHIP_EINVAL, "scatterND: shape missing");
  if (flags & ~(TFHIP_SCATTER_SUM | TFHIP_SCATTER_SKIP_INVALID | TFHIP_SCATTER_WIDE_SUM))
    return ctx->fail(TFHIP_EINVAL, "scatterND: unknown flag");
  Temp flat(ctx);
  int64_t slice = 0, rows = 0;
  int rc;
  // (row numbers that need no check are read as they are: a segment sum, two launches fewer)
  const bool skip = flags & TFHIP_SCATTER_SKIP_INVALID, as_they_are = skip && slice_rank == 1;
  if ((rc = flatten_checked(ctx, "scatterND", bi, out_shape, rank, num_updates, slice_rank, &flat, &slice, &rows,
                            !skip, as_they_are)))
    return rc;
  const bool scalar_update = bu->numel == 1 && num_updates * slice != 1;
  if (bo->numel != rows * slice || (!scalar_update && bu->numel != num_updates * slice))
    return ctx->fail(TFHIP_EINVAL, "scatterND: buffer sizes do not match the shapes given");
  if ((bo->dtype != TFHIP_FLOAT32 && bo->dtype != TFHIP_INT32) || bu->dtype != bo->dtype)
    return ctx->fail(TFHIP_EINVAL, "scatterND: updates and result must both be float32 or both int32");
  if (bo->numel == 0) return TFHIP_OK;
  if (rows > INT_MAX) return ctx->fail(TFHIP_ENOTSUP, "scatterND: more than 2^31 - 1 result slices");
  const int sum = flags & TFHIP_SCATTER_SUM ? 1 : 0, one = scalar_update ? 1 : 0;
  auto scatter = [&](const auto* fl) {
    if (bo->dtype == TFHIP_INT32)
      launch_scatter<int32_t, int32_t>(ctx, fl, (const int32_t*)bu->ptr, (int32_t*)bo->ptr, rows, slice, num_updates,
                                       (int32_t)default_value, sum, one);
    else if (flags & TFHIP_SCATTER_WIDE_SUM)
      launch_scatter<float, double>(ctx, fl, (const float*)bu->ptr, (float*)bo->ptr, rows, slice, num_updates,
                                    (float)default_value, sum, one);
    else
      launch_scatter<float, float>(ctx, fl, (const float*)bu->ptr, (float*)bo->ptr, rows, slice, num_updates,
                                   (float)default_value, sum, one);
  };
  if (as_they_are) scatter((const int32_t*)bi->ptr);
  else scatter((const int64_t*)flat.ptr);
  TFHIP_LAUNCH_CHECK(ctx);
  return TFHIP_OK;
}

extern "C" int tfhip_resize_bilinear_backprop(tfhip_ctx* ctx, int64_t dy, int64_t dx, int batch,
                                              int x_h, int x_w, int channels, int y_h, int y_w,
                                              int align_corners) {
  if (!ctx) return TFHIP_EINVAL;
  TFHIP_GET(ctx, bdy, dy);
  TFHIP_GET(ctx, bdx, dx);
  int rc;
  if ((rc = resize_backprop_check(ctx, "resizeBilinearBackprop", bdy, bdx, batch, x_h, x_w, channels, y_h, y_w)))
    return rc;
  if (bdx->numel == 0) return TFHIP_OK;
  // effective sizes and scales (backend_cpu.ts:2952-2963)
  const double eh_x = (align_corners && y_h > 1) ? x_h - 1 : x_h, ew_x = (align_corners && y_w > 1) ? x_w - 1 : x_w;
  const double eh_y = (align_corners && y_h > 1) ? y_h - 1 : y_h, ew_y = (align_corners && y_w > 1) ? y_w - 1 : y_w;
  if (bdy->numel == 0) return tfhip_fill(ctx, dx, 0.0);
  tfhip::launch(ctx, resize_bilinear_backprop_kernel, dim3(blocks_for(ctx, bdx->numel)), dim3(256), 0, (const float*)bdy->ptr, (float*)bdx->ptr, batch, x_h, x_w, channels,
                     y_h, y_w, eh_x / eh_y, ew_x / ew_y);
  TFHIP_LAUNCH_CHECK(ctx);
  return TFHIP_OK;
}

extern "C" int tfhip_resize_nearest_backprop(tfhip_ctx* ctx, int64_t dy, int64_t dx, int batch,
                                             int x_h, int x_w, int channels, int y_h, int y_w,
                                             int align_corners) {
  if (!ctx) return TFHIP_EINVAL;
  TFHIP_GET(ctx, bdy, dy);
  TFHIP_GET(ctx, bdx, dx);
  int rc;
  if ((rc = resize_backprop_check(ctx, "resizeNearestNeighborBackprop", bdy, bdx, batch, x_h, x_w, channels, y_h,
                                  y_w)))
    return rc;
  if (bdx->numel == 0) return TFHIP_OK;
  if (bdy->numel == 0) return tfhip_fill(ctx, dx, 0.0);
  // effective sizes and scales (backend_cpu.ts:3083-3094)
  const double eh_x = (align_corners && y_h > 1) ? x_h - 1 : x_h, ew_x = (align_corners && y_w > 1) ? x_w - 1 : x_w;
  const double eh_y = (align_corners && y_h > 1) ? y_h - 1 : y_h, ew_y = (align_corners && y_w > 1) ? y_w - 1 : y_w;
  tfhip::launch(ctx, resize_nearest_backprop_kernel, dim3(blocks_for(ctx, bdx->numel)), dim3(256), 0, (const float*)bdy->ptr, (float*)bdx->ptr, batch, x_h, x_w, channels,
                     y_h, y_w, eh_x / eh_y, ew_x / ew_y, align_corners ? 1 : 0);
  TFHIP_LAUNCH_CHECK(ctx);
  return TFHIP_OK;
}

extern "C" int tfhip_crop_and_resize(tfhip_ctx* ctx, int64_t images, int64_t boxes,
                                     int64_t box_index, int64_t out, int batch, int image_h,
                                     int image_w, int channels, int64_t num_boxes, int crop_h,
                                     int crop_w, int method, float extrapolation_value) {
  if (!ctx) return TFHIP_EINVAL;
  TFHIP_GET(ctx, bim, images);
  TFHIP_GET(ctx, bb, boxes);
  TFHIP_GET(ctx, bx, box_index);
  TFHIP_GET(ctx, bo, out);
  if (batch < 0 || image_h < 0 || image_w < 0 || channels < 0 || num_boxes < 0 || crop_h < 0 || crop_w < 0)
    return ctx->fail(TFHIP_EINVAL, "cropAndResize: bad geometry");
  if (method != TFHIP_RESIZE_BILINEAR && method != TFHIP_RESIZE_NEAREST)
    return ctx->fail(TFHIP_EINVAL, "cropAndResize: method must be bilinear or nearest");
  if (bim->numel != (int64_t)batch * image_h * image_w * channels || bb->numel != num_boxes * 4 ||
      bx->numel != num_boxes || bo->numel != num_boxes * crop_h * crop_w * channels)
    return ctx->fail(TFHIP_EINVAL, "cropAndResize: buffers do not match the shapes given");
  if (bb->dtype != TFHIP_FLOAT32 || bx->dtype != TFHIP_INT32 || bo->dtype != TFHIP_FLOAT32)
    return ctx->fail(TFHIP_EINVAL, "cropAndResize: boxes float32, box indices int32, result float32");
  if (bo->numel == 0) return TFHIP_OK;
  if (bim->numel == 0) return ctx->fail(TFHIP_EINVAL, "cropAndResize: empty image");
  Temp tx(ctx);
  const float* imf;
  int rc;
  if ((rc = as_f32(ctx, bim, &tx, &imf))) return rc;
  tfhip::launch(ctx, crop_and_resize_kernel, dim3(blocks_for(ctx, bo->numel)), dim3(256), 0,
                     imf, (const float*)bb->ptr, (const int32_t*)bx->ptr, (float*)bo->ptr, batch, image_h,
                     image_w, channels, num_boxes, crop_h, crop_w, method == TFHIP_RESIZE_NEAREST ? 1 : 0,
                     extrapolation_value);
  TFHIP_LAUNCH_CHECK(ctx);
  return TFHIP_OK;
}
