// Products of float32 matrices on the bf16 matrix cores, with the precision of float32.
//
// A float32 x is the exact sum of three bf16 values: h = x cut to 8 significant bits, m the rest
// rounded to 8, and what then remains has at most 8 bits left, which is l.  bf16 has the
// exponents of float32, and the product of two bf16 values is exact in float32, so
//   a * b = ah bh + (ah bm + am bh) + (ah bl + am bm + al bh)
// up to terms below 2^-22 of it and of either sign.  Six bf16 matrix instructions (32 x 32 x 16, 1024
// flop per clock and SIMD) then do what eight float32 ones (32 x 32 x 2, 64 flop per clock) do.
//
// Kernel shape.  WM x WN wavefronts own a BM x BN tile, each TM x 2 accumulators of 32 x 32.  K is
// walked 16 at a time through two LDS buffers; an element is split once per workgroup that reads
// it, on its way from registers into LDS, between the matrix instructions of the step before.
//
// What bounds it: a 128 x 128 step is 24 matrix instructions per wavefront, 19 ns each with
// nothing else in the machine and 23.6 with the six vector instructions per matrix instruction
// that splitting and addressing cost, and takes 34; LDS is busy a quarter of the time, without
// conflicts.  Gradients of 3 x 3 convolutions run at 93 to 153 TFLOP/s (float32 kernels 63 to 99, and
// 157 is the float32 matrix peak).  Measured without effect on that: one buffer of 32 k, loads two
// steps ahead, the leading parts read before the barrier, v_cvt_pk_bf16_f32 for the splits.
//
// LDS layout.  Per operand three planes (h, m, l) of [k / 8][slot][8 bf16]: the matrix instruction
// takes 8 consecutive k of a row per lane, and 32 lanes read 512 consecutive bytes.  A slot is a
// row of A or a column of B; where the operand lies with rows (columns) contiguous in memory a
// thread takes 2 k x 4 rows and turns them around in registers, and the slots of 64 rows are
// dealt so that the 4 rows of a thread go to 4 runs of 16 slots (see slot_of): without that the
// writes of a wavefront would meet in a quarter of the banks.
//
// Special values.  An infinity makes every sum it enters NaN here (its rest is infinity minus
// infinity), and of a value below 2^-110 the last bits can lie below 2^-133, the smallest bf16.  So
// a workgroup that finds a result that is not finite, or that has staged an operand which is not
// the sum of its parts, computes its tile again with float32 matrix instructions, and the result
// is what the float32 kernels give.  Such a tile takes the time of both: [4096, 1024]^T-shaped x
// [1024, 1024] 78 us, 157 with one infinity or one value of 2^-120 (float32 kernels 93).  Small
// results need nothing of the kind: these instructions take and give denormal values, and with
// both operands near 2^-63 the error is 0.7e-7 here and 0.9e-7 there.
#include <type_traits>

#include "tfhip_gemm.h"

namespace tfhip {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

constexpr int SK = 16;           // k per step
constexpr int SPLIT_PLAIN_K = 128;  // matMul: longer ranges of K are summed in blocks
constexpr int SPLIT_BLOCK = 8;      // of this many steps
// Fewer products than this stay in float32, which rounds once per product or two: the largest error
// seen over 4 to 17 M results, in 2^-24 of the products' magnitudes, float32 kernels and these: K = 1
// 1.0 and 4.1, 2 1.9 and 4.1, 3 2.8 and 3.6, 4 3.2 and 3.6, 5 3.5 and 3.3, 8 4.3 and 2.6; relative
// (2-norm) 2.5e-8 and 3.1e-8, 3.1 and 3.1, 3.6 and 3.2, 4.0 and 3.2, 4.4 and 3.2, 5.4 and 3.2.
constexpr int SPLIT_LEAST_K = 5;
constexpr int SPLIT_FOLD = 4;       // steps per block where a tile is summed in float32

// The slot of row (column) r of a tile and its inverse: within 64, row 4c + e goes to slot
// 32 (e & 1) + 16 (e >> 1) + c.  A lane that holds the same slot of two neighbouring accumulators
// holds two neighbouring columns, and 32 lanes cover 64 columns.
__device__ __forceinline__ int slot_of(int r) {
  return (r & ~63) + (r & 1) * 32 + ((r >> 1) & 1) * 16 + ((r >> 2) & 15);
}
__device__ __forceinline__ int row_of(int s) {
  return (s & ~63) + 4 * (s & 15) + 2 * ((s >> 4) & 1) + ((s >> 5) & 1);
}

// Two consecutive k as three bf16 pairs.  h is x cut to 8 significant bits, m what is left rounded
// to 8 (so that l, and with it the products left out, has either sign), l the rest: x = h + m + l
// exactly.  Integer operations and byte permutes (v_dot2_f32_bf16, which would subtract without
// unpacking, is slower).  What l leaves are bits below the upper half of the last rest: `lost`
// collects that word of every value, at one instruction for two: 3 x [1280, 1600] x [1600, 2240]
// takes 220 us without and 224 with it (243 with a running minimum of the magnitudes, three
// instructions for two).
__device__ __forceinline__ void split2(float x0, float x1, unsigned& h, unsigned& m, unsigned& l, unsigned& lost) {
  constexpr unsigned TOP = 0x07060302u;  // the upper halves of two words as one
  auto top = [](unsigned u) { return __builtin_bit_cast(float, u & 0xffff0000u); };
  const unsigned u0 = __builtin_bit_cast(unsigned, x0), u1 = __builtin_bit_cast(unsigned, x1);
  h = __builtin_amdgcn_perm(u1, u0, TOP);
  const float r0 = x0 - top(u0), r1 = x1 - top(u1);
  const unsigned v0 = __builtin_bit_cast(unsigned, r0) + 0x8000u, v1 = __builtin_bit_cast(unsigned, r1) + 0x8000u;
  m = __builtin_amdgcn_perm(v1, v0, TOP);
  const unsigned w0 = __builtin_bit_cast(unsigned, r0 - top(v0)), w1 = __builtin_bit_cast(unsigned, r1 - top(v1));
  l = __builtin_amdgcn_perm(w1, w0, TOP);
  // (as one instruction here and now: as an expression the compiler keeps the words and joins them
  // later, which took up to 17 registers)
  asm("v_or3_b32 %0, %1, %2, %0" : "+v"(lost) : "v"(w0), "v"(w1));
}

template <int WM_, int WN_, int TM_>
struct SplitCfg {
  static constexpr int WM = WM_, WN = WN_, TM = TM_, TN = 2;
  static constexpr int BM = WM * TM * 32, BN = WN * TN * 32, THREADS = WM * WN * 64;
};

// How one operand's tile of ROWS x 16 is staged: by items of 4 k of a row (k contiguous in
// memory) or of 2 k x 4 rows (rows contiguous), REGS vectors of 4 per thread.  Where there are
// fewer items than threads two threads stage the same one.
template <int ROWS, int THREADS, bool KC_>
struct Staging {
  static constexpr int ITEMS = KC_ ? ROWS * 4 : ROWS * 2;
  static constexpr int PER = (ITEMS + THREADS - 1) / THREADS;
  static constexpr bool KC = KC_;
  static constexpr int REGS = KC ? PER : 2 * PER;
  static constexpr int GROUP = ROWS * 16 + 64;  // bytes from one k / 8 to the next: 64 spare ones
  static constexpr int PLANE = 2 * GROUP;       // so that the two lie in different banks
  // row and k of item `i` of this thread within the tile; a row of k-contiguous items is a slot
  static __device__ __forceinline__ int row(int tid, int i) {
    const int item = (tid + i * THREADS) % ITEMS;
    return KC ? item / 4 : ((item >> 2) % (ROWS / 4)) * 4;
  }
  static __device__ __forceinline__ int k(int tid, int i) {
    const int item = (tid + i * THREADS) % ITEMS;
    return KC ? (item & 3) * 4 : (item / ROWS) * 8 + (item & 3) * 2;
  }
};

// `hi` adds up the products of the leading parts and `lo` the others, 2^-8 of it, so that the sum
// is rounded once per 16 k.  (In one sum the small products lose their last bits to the large
// total, always downwards: measured with K = 256 signed values, 1.4e-7 relative with a bias of
// -6e-9 against 0.8e-7 without one.)  BLOCKED > 0: `hi` starts from zero every BLOCKED steps and
// joins a total of its own, for sums so long that one rounding per 16 k of the whole would be
// more than the two-level sum of the float32 kernels shows.  Measured against 64 bits, float32
// kernels and these: matMul of signed values with K = 128 1.25e-7 and 0.62e-7, 1024 1.54e-7 and
// 0.83e-7 (1.63e-7 without blocks), 4096 2.1e-7 and 1.2e-7; of positive ones 0.69 and 0.62, 0.72
// and 0.56, 1.26 and 0.82; gradients of convolutions 2.2e-7 to 7.1e-7 and 1.1e-7 to 2.3e-7.  What is
// left out shows where there are few products (see SPLIT_LEAST_K).
template <class T, int AMODE, int BMODE, int BLOCKED, bool VEC>
__global__ __launch_bounds__(T::THREADS, 2) void gemm_split_kernel(const GemmArgs p) {
  constexpr int BM = T::BM, BN = T::BN, TM = T::TM, TN = T::TN, THREADS = T::THREADS;
  constexpr bool A_KC = AMODE == A_ROWMAJOR || AMODE == A_IM2COL || AMODE == A_IM2COL_TAPS;
  constexpr bool B_KC = BMODE == B_TRANSPOSED;
  static_assert(BM % 64 == 0 && BN % 64 == 0, "slots are dealt within 64 rows");
  using SA = Staging<BM, THREADS, A_KC>;
  using SB = Staging<BN, THREADS, B_KC>;
  constexpr int BUF = 3 * SA::PLANE + 3 * SB::PLANE;
  __shared__ __attribute__((aligned(16))) char lds[2 * BUF];
  static_assert(BM * 64 + BN * 64 <= BUF, "room for float32 operands");
  __shared__ int redo_of[T::WM * T::WN];

  const int tid = threadIdx.x;
  __builtin_assume(tid >= 0 && tid < THREADS);
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / T::WN, wn = wave % T::WN;
  const int l32 = lane & 31, g = lane >> 5;

  const WorkItem cur = work_item(p, blockIdx.x);
  if (cur.tile < 0) return;
  const int tiles_per_batch = p.tiles_m * p.tiles_n;
  const int batch = cur.tile < tiles_per_batch ? 0 : cur.tile / tiles_per_batch;
  int tm, tn;
  tile_row_col(p, cur.tile - batch * tiles_per_batch, tm, tn);
  const int bm0 = tm * BM, bn0 = tn * BN;
  const __amdgpu_buffer_rsrc_t ra = make_rsrc(p.A + batch * p.strideA, p.a_bytes);
  const __amdgpu_buffer_rsrc_t rb = make_rsrc(static_cast<const float*>(p.B) + batch * p.strideB, p.b_bytes);

  // ---- what this thread stages ----
  unsigned a_at[SA::PER], b_at[SB::PER];  // byte offset of the item at k = 0; OOB_OFFSET: no such row
  int a_ih[SA::PER], a_iw[SA::PER];       // gathers: image row and column at the first tap (pixel)
  unsigned a_taps[SA::PER];               // A_IM2COL_TAPS: the taps inside the image, a bit each
  // Position of the thread's next k in a gather: channel and filter column (A_IM2COL), or output
  // column and output row (A_IM2COL_T); the image rows, columns and bytes it lies from where the
  // item starts, kept up by additions (a 32-bit multiply takes four times an addition's time).
  int g_inner = 0, g_middle = 0, g_row = 0, g_col = 0;
  unsigned g_at = 0;
  int k_next = 0;
  auto setup = [&]() {
    k_next = cur.kt0 * SK;
#pragma unroll
    for (int i = 0; i < SA::PER; i++) {
      a_ih[i] = a_iw[i] = 0;
      const int row = bm0 + SA::row(tid, i);
      const bool ok = row < p.M;
      if (AMODE == A_ROWMAJOR) {
        a_at[i] = ok ? ((unsigned)row * p.lda + SA::k(tid, 0)) * 4u : OOB_OFFSET;
      } else if (AMODE == A_TRANSPOSED) {
        a_at[i] = ok ? ((unsigned)SA::k(tid, i) * p.lda + row) * 4u : OOB_OFFSET;
      } else if (AMODE == A_IM2COL) {
        const int ow = row % p.OW, r = row / p.OW;
        const int oh = r % p.OH, n = r / p.OH;
        a_ih[i] = ok ? oh * p.sh - p.pt : -0x40000000;  // (a row past the last: no image row)
        a_iw[i] = ow * p.sw - p.pl;
        a_at[i] = (unsigned)((n * p.H + a_ih[i]) * p.W + a_iw[i]) * p.Cin * 4u;
      } else if (AMODE == A_IM2COL_TAPS) {
        const int ow = row % p.OW, r = row / p.OW;
        const int oh = r % p.OH, n = r / p.OH;
        const int ih = oh * p.sh - p.pt, iw = ow * p.sw - p.pl;
        unsigned columns = 0, taps = 0;
        for (int kw = 0; kw < p.KW; kw++) columns |= ((unsigned)(iw + kw * p.dw) < (unsigned)p.W ? 1u : 0u) << kw;
        for (int kh = 0; kh < p.KH; kh++)
          taps |= ((unsigned)(ih + kh * p.dh) < (unsigned)p.H ? columns : 0u) << (kh * p.KW);
        a_taps[i] = ok ? taps : 0u;
        a_at[i] = ((unsigned)((n * p.H + ih) * p.W + iw) * p.Cin + SA::k(tid, 0)) * 4u;
      } else {
        const int tap = row / p.Cin, c = row - tap * p.Cin;
        const int kh = tap / p.KW, kw = tap - kh * p.KW;
        a_ih[i] = ok ? kh * p.dh - p.pt : -0x40000000;
        a_iw[i] = kw * p.dw - p.pl;
        a_at[i] = (unsigned)((a_ih[i] * p.W + a_iw[i]) * p.Cin + c) * 4u;
      }
    }
    const int k = k_next + SA::k(tid, 0);
    if (AMODE == A_IM2COL) {
      const int tap = k / p.Cin, kh = tap / p.KW;
      g_inner = k - tap * p.Cin;
      g_middle = tap - kh * p.KW;
      g_row = kh * p.dh;
      g_col = g_middle * p.dw;
      g_at = (unsigned)((g_row * p.W + g_col) * p.Cin + g_inner) * 4u;
    }
    if (AMODE == A_IM2COL_T) {
      const int r = k / p.OW, n = r / p.OH;
      g_inner = k - r * p.OW;
      g_middle = r - n * p.OH;
      g_row = g_middle * p.sh;
      g_col = g_inner * p.sw;
      g_at = (unsigned)((n * p.H + g_row) * p.W + g_col) * p.Cin * 4u;
    }
#pragma unroll
    for (int i = 0; i < SB::PER; i++) {
      const int col = bn0 + (B_KC ? row_of(SB::row(tid, i)) : SB::row(tid, i));
      const bool ok = col < p.N;
      b_at[i] = ok ? (B_KC ? (unsigned)col * p.ldb + SB::k(tid, 0) : (unsigned)SB::k(tid, i) * p.ldb + col) * 4u
                   : OOB_OFFSET;
    }
  };

  // 4 consecutive elements, at 4-byte alignment where rows are not whole vectors: the hardware takes
  // that, and checks the range of each of the four (four loads of 4 bytes: [3001, 1000] x [1000, 3001],
  // both turned, 363 us, 158 like this, 250 in float32).  `base` is the same for all lanes; the
  // range check is on the sum.
  auto load4 = [&](const __amdgpu_buffer_rsrc_t& r, unsigned at, int base) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)at, base, 0));
  };
  struct Raw {
    f32x4 a[SA::REGS], b[SB::REGS];
    int a_left, b_left;  // unaligned rows along k: how many of a vector's k there are
  };
  // What follows the last k of a row in memory is another row.  (Rows or columns past the last in a
  // vector along them are harmless: their products are not stored.)
  auto trim = [&](f32x4 v, int left) {
#pragma unroll
    for (int e = 1; e < 4; e++) v[e] = e < left ? v[e] : 0.f;
    return v;
  };
  // From one output pixel to the next row's first, and from an image's last to the next image.
  const unsigned to_row = AMODE == A_IM2COL ? (unsigned)(p.dh * p.W - p.KW * p.dw) * p.Cin * 4u
                                            : (unsigned)(p.sh * p.W - p.OW * p.sw) * p.Cin * 4u;
  const unsigned to_image = (unsigned)(p.H - p.OH * p.sh) * p.W * p.Cin * 4u;
  // The next step's operands on their way into registers: no branches, so that the matrix
  // instructions can go between.  Steps past the last one of a range read what lies there, and
  // zeros past K; nobody multiplies them.  (Rows at or beyond K of an operand whose rows lie along
  // K are out of its range by themselves.)
  auto load = [&](Raw& o) {
    const int k0 = __builtin_amdgcn_readfirstlane(k_next);
    if (AMODE == A_ROWMAJOR) {
      o.a_left = p.K - k0 - SA::k(tid, 0);  // (the same for all items of a thread)
#pragma unroll
      for (int i = 0; i < SA::PER; i++) o.a[i] = load4(ra, o.a_left > 0 ? a_at[i] : OOB_OFFSET, k0 * 4);
    } else if (AMODE == A_IM2COL) {
      // (the 4 channels of an item share a filter tap: Cin is a multiple of 4)
      const bool in_k = k0 + SA::k(tid, 0) < p.K;
#pragma unroll
      for (int i = 0; i < SA::PER; i++) {
        const bool ok = in_k & ((unsigned)(a_ih[i] + g_row) < (unsigned)p.H) &
                        ((unsigned)(a_iw[i] + g_col) < (unsigned)p.W);
        o.a[i] = buffer_load_f32x4(ra, ok ? a_at[i] + g_at : OOB_OFFSET);
      }
    } else if (AMODE == A_IM2COL_TAPS) {
      // (a step lies in one tap: its place is scalar arithmetic, a look at a bit says whether it is there)
      const unsigned tap = p.by_cin.quotient((unsigned)k0), kh = p.by_kw.quotient(tap);
      const unsigned at = (((kh * p.dh) * p.W + (tap - kh * p.KW) * p.dw) * p.Cin + (k0 - tap * p.Cin)) * 4u;
      const unsigned bit = k0 < p.K ? 1u << tap : 0u;
#pragma unroll
      for (int i = 0; i < SA::PER; i++) o.a[i] = buffer_load_f32x4(ra, a_taps[i] & bit ? a_at[i] + at : OOB_OFFSET);
    } else if (AMODE == A_TRANSPOSED) {
#pragma unroll
      for (int i = 0; i < SA::PER; i++)
#pragma unroll
        for (int e = 0; e < 2; e++) o.a[2 * i + e] = load4(ra, a_at[i], (k0 + e) * p.lda * 4);
    } else {
      static_assert(AMODE != A_IM2COL_T || SA::PER == 1, "one pixel position per thread");
      const int k = k0 + SA::k(tid, 0);
      const bool wrap = g_inner + 1 == p.OW, wrap_image = wrap & (g_middle + 1 == p.OH);
      const int row1 = wrap_image ? 0 : wrap ? g_row + p.sh : g_row, col1 = wrap ? 0 : g_col + p.sw;
      const unsigned at1 = g_at + (unsigned)p.sw * p.Cin * 4u + (wrap ? to_row : 0u) + (wrap_image ? to_image : 0u);
#pragma unroll
      for (int e = 0; e < 2; e++) {
        const bool ok = (k + e < p.K) & ((unsigned)(a_ih[0] + (e ? row1 : g_row)) < (unsigned)p.H) &
                        ((unsigned)(a_iw[0] + (e ? col1 : g_col)) < (unsigned)p.W);
        o.a[e] = buffer_load_f32x4(ra, ok ? a_at[0] + (e ? at1 : g_at) : OOB_OFFSET);
      }
    }
    if (B_KC) {
      o.b_left = p.K - k0 - SB::k(tid, 0);
#pragma unroll
      for (int i = 0; i < SB::PER; i++) o.b[i] = load4(rb, o.b_left > 0 ? b_at[i] : OOB_OFFSET, k0 * 4);
    } else {
#pragma unroll
      for (int i = 0; i < SB::PER; i++)
#pragma unroll
        for (int e = 0; e < 2; e++) o.b[2 * i + e] = load4(rb, b_at[i], (k0 + e) * p.ldb * 4);
    }
  };
  auto advance = [&]() {
    k_next += SK;
    if (AMODE == A_IM2COL) {
      g_inner += SK;
      g_at += SK * 4;
      while (g_inner >= p.Cin) {
        g_inner -= p.Cin;
        g_col += p.dw;
        g_at += (unsigned)(p.dw - 1) * p.Cin * 4u;
        if (++g_middle == p.KW) {
          g_middle = 0;
          g_col = 0;
          g_row += p.dh;
          g_at += to_row;
        }
      }
    }
    if (AMODE == A_IM2COL_T) {
      g_inner += SK;
      g_col += SK * p.sw;
      g_at += (unsigned)(SK * p.sw) * p.Cin * 4u;
      while (g_inner >= p.OW) {
        g_inner -= p.OW;
        g_col -= p.OW * p.sw;
        g_row += p.sh;
        g_at += to_row;
        if (++g_middle == p.OH) {
          g_middle = 0;
          g_row = 0;
          g_at += to_image;
        }
      }
    }
  };

  // ---- registers -> LDS ----
  unsigned lost = 0;  // (see split2) of the operands this thread has staged
  // An operand's items go into its planes at `base` in pieces of one split each: piece 2i + j is
  // the j-th pair of k of item i (k contiguous; the second writes both), piece 4i + e the pair of
  // k of row e of item i.
  auto put_piece = [&](auto staging_tag, char* base, const f32x4* v, int left, unsigned (&half)[3], int n) {
    using S = decltype(staging_tag);
    unsigned part[3];
    if (S::KC) {
      const int i = n / 2, row = S::row(tid, i), k = S::k(tid, i);
      const f32x4 x = VEC ? v[i] : trim(v[i], left);
      split2(x[2 * (n & 1)], x[2 * (n & 1) + 1], part[0], part[1], part[2], lost);
      char* at = base + (k >> 3) * S::GROUP + row * 16 + (k & 4) * 2;
#pragma unroll
      for (int s = 0; s < 3; s++) {
        if (n & 1) *reinterpret_cast<u32x2*>(at + s * S::PLANE) = u32x2{half[s], part[s]};
        else half[s] = part[s];
      }
    } else {
      // (slot_of(row + e): row is 4c)
      const int i = n / 4, e = n & 3, slot = slot_of(S::row(tid, i)) + (e & 1) * 32 + (e >> 1) * 16, k = S::k(tid, i);
      split2(v[2 * i][e], v[2 * i + 1][e], part[0], part[1], part[2], lost);
      char* at = base + (k >> 3) * S::GROUP + slot * 16 + (k & 6) * 2;
#pragma unroll
      for (int s = 0; s < 3; s++) *reinterpret_cast<unsigned*>(at + s * S::PLANE) = part[s];
    }
  };
  constexpr int A_PIECES = SA::REGS * 2, B_PIECES = SB::REGS * 2;
  unsigned half[3];
  auto stage_piece = [&](char* buf, const Raw& o, int n) {
    if (n < A_PIECES) put_piece(SA(), buf, o.a, o.a_left, half, n);
    else put_piece(SB(), buf + 3 * SA::PLANE, o.b, o.b_left, half, n - A_PIECES);
  };
  // The same as float32 [k / 4][slot][4].
  auto put_exact = [&](auto staging_tag, char* base, const f32x4* v, int left) {
    using S = decltype(staging_tag);
#pragma unroll
    for (int i = 0; i < S::PER; i++) {
      const int row = S::row(tid, i), k = S::k(tid, i);
      if (S::KC) {
        *reinterpret_cast<f32x4*>(base + (k >> 2) * (S::GROUP - 64) + row * 16) = VEC ? v[i] : trim(v[i], left);
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
          *reinterpret_cast<f32x2*>(base + (k >> 2) * (S::GROUP - 64) + slot_of(row + e) * 16 + (k & 2) * 4) =
              f32x2{v[2 * i][e], v[2 * i + 1][e]};
      }
    }
  };
  f32x16 hi[TM][TN], lo[TM][TN], total[TM][TN];
  const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  auto clear = [&](f32x16 (&sum)[TM][TN]) {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++) sum[i][j] = zero;
  };
  auto add = [&](f32x16 (&to)[TM][TN], const f32x16 (&x)[TM][TN]) {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++) to[i][j] += x[i][j];
  };
  const int a_slot = (wm * TM * 32 + l32) * 16, b_slot = (wn * TN * 32 + l32) * 16;

  clear(hi);
  clear(lo);
  if (BLOCKED) clear(total);
  setup();
  {
    struct Frags {
      bf16x8 a[TM], b[TN];
    };
    auto read = [&](const char* buf, int plane, Frags& f) {
#pragma unroll
      for (int i = 0; i < TM; i++)
        f.a[i] = *reinterpret_cast<const bf16x8*>(buf + plane * SA::PLANE + g * SA::GROUP + a_slot + i * 512);
#pragma unroll
      for (int j = 0; j < TN; j++)
        f.b[j] = *reinterpret_cast<const bf16x8*>(buf + 3 * SA::PLANE + plane * SB::PLANE + g * SB::GROUP + b_slot + j * 512);
    };
    // One step, for the tile in `buf`, whose leading parts `fh` are in registers on entry:
    //   read the other parts                (latency behind the first products)
    //   two thirds of the products; between them the next tile, in `raw`, goes split into `other`,
    //   and the loads of the one after it are issued
    //   barrier                             (the next tile is visible)
    //   read the next tile's leading parts  (latency behind the other products)
    //   the other products
    // so that the matrix cores have work on both sides of the barrier, and the vector ALU splits
    // while they multiply.  sched_barrier(0) pins that order: left alone, the scheduler gathers
    // all splits in front of all products.
    auto step = [&](const char* buf, char* other, Raw& raw, const Frags& fh, Frags& next) {
      Frags fm, fl;
      constexpr int PER_PRODUCT = TM * TN, BEFORE = 4 * PER_PRODUCT, PIECES = A_PIECES + B_PIECES;
      auto multiply = [&](int n) {  // matrix instruction n of the step
        const int s = n / PER_PRODUCT, i = n % PER_PRODUCT / TN, j = n % TN;
        const Frags& x = s == 2 || s == 3 ? fm : s == 5 ? fl : fh;
        const Frags& y = s == 1 || s == 3 ? fm : s == 4 ? fl : fh;
        f32x16& sum = s > 0 ? lo[i][j] : hi[i][j];
        sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x.a[i], y.b[j], sum, 0, 0, 0);
      };
      advance();
      read(buf, 1, fm);
      read(buf, 2, fl);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < BEFORE; n++) {
        multiply(n);
#pragma unroll
        for (int t = n * PIECES / BEFORE; t < (n + 1) * PIECES / BEFORE; t++) stage_piece(other, raw, t);
        if (n == BEFORE - 1) load(raw);
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();
      read(other, 0, next);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = BEFORE; n < 6 * PER_PRODUCT; n++) multiply(n);
      __builtin_amdgcn_sched_barrier(0);
    };
    Raw raw;
    Frags f0, f1;
    load(raw);
    advance();
#pragma unroll
    for (int t = 0; t < A_PIECES + B_PIECES; t++) stage_piece(lds, raw, t);
    load(raw);
    __syncthreads();
    read(lds, 0, f0);
    for (int kt = cur.kt0; kt < cur.kt1; kt += 2) {
      step(lds, lds + BUF, raw, f0, f1);
      if (kt + 1 < cur.kt1) step(lds + BUF, lds, raw, f1, f0);
      if (BLOCKED && ((kt - cur.kt0) & (BLOCKED - 1)) == BLOCKED - 2) {
        add(total, hi);
        clear(hi);
      }
    }
    if (BLOCKED) add(hi, total);
    add(hi, lo);
  }
  {
    // (zero times what is not finite is NaN, and so is every sum with it: one instruction a value)
    float zeros[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) zeros[r & 3] = __builtin_fmaf(hi[i][j][r], 0.f, zeros[r & 3]);
    const bool redo = (lost & 0xffffu) != 0 || !((zeros[0] + zeros[1]) + (zeros[2] + zeros[3]) == 0.f);
    // (the whole workgroup takes the branch or none of it does: it holds barriers)
    const int any_lane = __any(redo) ? 1 : 0;
    if (lane == 0) redo_of[wave] = any_lane;
    __syncthreads();
    int any_wave = 0;
#pragma unroll
    for (int i = 0; i < T::WM * T::WN; i++) any_wave |= redo_of[i];
    if (__builtin_amdgcn_readfirstlane(any_wave)) {
      // Again in float32: lanes 0..31 take k quad 2q, the others 2q + 1, the same for both operands.
      clear(hi);
      clear(lo);
      setup();
      Raw raw;
      for (int kt = cur.kt0; kt < cur.kt1; kt++) {
        load(raw);
        advance();
        put_exact(SA(), lds, raw.a, raw.a_left);
        put_exact(SB(), lds + BM * 64, raw.b, raw.b_left);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < SK / 8; q++) {
          f32x4 af[TM], bf[TN];
#pragma unroll
          for (int i = 0; i < TM; i++)
            af[i] = *reinterpret_cast<const f32x4*>(lds + (2 * q + g) * (SA::GROUP - 64) + a_slot + i * 512);
#pragma unroll
          for (int j = 0; j < TN; j++)
            bf[j] = *reinterpret_cast<const f32x4*>(lds + BM * 64 + (2 * q + g) * (SB::GROUP - 64) + b_slot + j * 512);
#pragma unroll
          for (int e = 0; e < 4; e++)
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
              for (int j = 0; j < TN; j++)
                lo[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[i][e], bf[j][e], lo[i][j], 0, 0, 0);
        }
        __syncthreads();
        if (((kt - cur.kt0) & (SPLIT_FOLD - 1)) == SPLIT_FOLD - 1) {
          add(hi, lo);
          clear(lo);
        }
      }
      add(hi, lo);
    }
  }

  // ---- store: register r of an accumulator holds slot 8 (r / 4) + 4 g + r % 4 of its rows; the
  // two accumulators of a row hold columns col and col + 1 ----
  const int lcol = row_of(wn * 64 + l32), col = bn0 + lcol;
  auto local_row = [&](int i, int r) {
    const int s = wm * TM * 32 + i * 32 + 8 * (r >> 2) + 4 * g + (r & 3);
    return A_KC ? s : row_of(s);
  };
  if (cur.slot >= 0) {
    float* slot = p.partials + (long long)cur.slot * (BM * BN) + lcol;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int r = 0; r < 16; r++)
        *reinterpret_cast<f32x2*>(slot + local_row(i, r) * BN) = f32x2{hi[i][0][r], hi[i][1][r]};
    return;
  }
  float bias_c[TN] = {0.f, 0.f}, alpha_c[TN] = {0.f, 0.f};
#pragma unroll
  for (int j = 0; j < TN; j++) {
    if (p.bias_kind == TFHIP_BCAST_SCALAR) bias_c[j] = p.bias[0];
    if (p.bias_kind == TFHIP_BCAST_COLUMN && col + j < p.N) bias_c[j] = p.bias[col + j];
    if (p.prelu_kind == TFHIP_BCAST_SCALAR) alpha_c[j] = p.prelu[0];
    if (p.prelu_kind == TFHIP_BCAST_COLUMN && col + j < p.N) alpha_c[j] = p.prelu[col + j];
  }
  const long long tile_at = batch * p.strideC + (long long)bm0 * p.N + bn0;
  const bool full_bias = p.bias_kind == TFHIP_BCAST_FULL, full_alpha = p.prelu_kind == TFHIP_BCAST_FULL;
  if (full_bias || full_alpha || p.act == TFHIP_ACT_PRELU) {
    const ActCfg act = act_cfg(p.act);
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int r = 0; r < 16; r++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
          const int row = local_row(i, r);
          if (bm0 + row >= p.M || col + j >= p.N) continue;
          const long long at = tile_at + (long long)row * p.N + lcol + j;
          const float bv = full_bias ? p.bias[at] : bias_c[j];
          const float al = full_alpha ? p.prelu[at] : alpha_c[j];
          p.C[at] = activate(hi[i][j][r] + bv, act, al);
        }
    return;
  }
  // (32-bit offsets: the planner keeps BM * N below 2^29 elements.  Written through the L2: see
  // STORE_WRITE_THROUGH.)
  const Clamp cl = clamp_of(p.act);
  const __amdgpu_buffer_rsrc_t rc = make_rsrc(p.C + tile_at, 0x7fffffffu);
  auto store = [&](auto put) {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int row = local_row(i, r);
        const bool in = bm0 + row < p.M && col < p.N;
        const float v0 = clamp(hi[i][0][r] + bias_c[0], cl), v1 = clamp(hi[i][1][r] + bias_c[1], cl);
        put(in ? (unsigned)(row * p.N + lcol) * 4u : OOB_OFFSET,
            u32x2{__builtin_bit_cast(unsigned, v0), __builtin_bit_cast(unsigned, v1)});
      }
  };
  if ((p.N & 1) == 0) {
    store([&](unsigned at, u32x2 v) { __builtin_amdgcn_raw_buffer_store_b64(v, rc, (int)at, 0, STORE_WRITE_THROUGH); });
    return;
  }
  // N odd: pairs of columns at 4-byte alignment, and the last column by itself.  Rows share their
  // cache lines with their neighbours, so these stores wait in the L2 to be put together.  (Two
  // 4-byte stores written through: 22 x [491, 16] x [16, 805] 24.4 us, 15.8 like this.)
  const bool last = col + 1 == p.N, has_last = bn0 + BN >= p.N;
  store([&](unsigned at, u32x2 v) {
    __builtin_amdgcn_raw_buffer_store_b64(v, rc, (int)(last ? OOB_OFFSET : at), 0, 0);
    if (has_last) __builtin_amdgcn_raw_buffer_store_b32(v[0], rc, (int)(last ? at : OOB_OFFSET), 0, 0);
  });
}

// ---------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------
struct SplitPlan {
  int cfg = -1, tiles_m = 0, tiles_n = 0, full = 0, tail = 0, splits = 1, kt_per = 0;
  double cost = 0;
};

// The best plan of one tile shape, against `best`, by an estimate in microseconds: a launch, and
// the steps of the busiest CU.  A step of a workgroup alone on its CU takes `alone` us and one of
// several `shared` (measured: [128, 128] tiles 0.80 and 0.80, their wavefronts fill a CU; [64, 128]
// 0.56 and 0.48; [128, 64] 0.60 and 0.58; [256, 64] 1.20 and 0.88, which is a quarter less than two of the
// former: where there are at most 64 columns a wavefront of 64 x 64 splits and reads from LDS
// two thirds of what two of 32 x 64 do).  A cut along K costs a second launch and the partial
// tiles' way through memory.  `most_steps`: longest range of K the shape may be given.
static void plan_cfg(SplitPlan& best, int cfg, int bm, int bn, double alone, double shared, int most_steps,
                     const GemmArgs& p, int batch, int cus) {
  SplitPlan pl;
  pl.cfg = cfg;
  pl.tiles_m = (int)ceil_div(p.M, bm);
  pl.tiles_n = (int)ceil_div(p.N, bn);
  const long long tiles = (long long)pl.tiles_m * pl.tiles_n * batch;
  const int k_tiles = (int)ceil_div(p.K, SK);
  if (tiles > 0x3fffffff) return;
  // (several per CU: whole rounds, or half a one more where many follow each other freely)
  auto rounds = [&](long long items, int steps) {
    const double n = (double)items / cus, up = (double)ceil_div(items, cus);
    return steps * (items <= cus ? alone : shared * (up < n + 0.5 ? up : n + 0.5));
  };
  auto offer = [&](const SplitPlan& sp) {
    if (best.cfg < 0 || sp.cost < best.cost) best = sp;
  };
  pl.full = (int)tiles;
  pl.kt_per = k_tiles;
  pl.cost = 4.0 + rounds(tiles, k_tiles);
  if (k_tiles <= most_steps) offer(pl);
  if (k_tiles < 16) return;
  // every tile cut along K, or those that are left after whole rounds
  for (const long long cut_tiles : {tiles < 2 * cus ? tiles : 0, tiles > cus ? tiles % cus : 0}) {
    if (cut_tiles == 0 || (cut_tiles < tiles && k_tiles > most_steps)) continue;
    for (int want = 2; want <= 4 * cus / (int)cut_tiles; want++) {
      SplitPlan sp = pl;
      sp.kt_per = (int)ceil_div(ceil_div(k_tiles, want), 2) * 2;
      if (sp.kt_per < 8) break;
      if (sp.kt_per > most_steps) continue;
      sp.splits = (int)ceil_div(k_tiles, sp.kt_per);
      if (sp.splits < 2) continue;
      sp.tail = (int)cut_tiles;
      sp.full = (int)(tiles - cut_tiles);
      const long long items = cut_tiles * sp.splits;
      sp.cost = 4.0 + (sp.full ? shared * k_tiles * (sp.full / cus) : 0.0) + rounds(items, sp.kt_per) + 4.5 +
                2.0 * items * (double)bm * bn * 4 / 5.0e6;
      offer(sp);
    }
  }
}

// The same estimate for the float32 kernels in 64 x 64 tiles: 0.4 us for a step of 16 k where the
// grid is sparse, 0.33 us per tile where it is full (100 TFLOP/s), more where the operands are
// turned around or gathered; and their cut along K.
static double float32_cost(const GemmArgs& p, int batch, int cus, int amode, int bmode) {
  const double tiles = (double)ceil_div(p.M, 64) * (double)ceil_div(p.N, 64) * batch;
  const double steps = (double)ceil_div(p.K, 16);
  const double slower = amode == A_IM2COL_UP ? 1.35 : amode == A_IM2COL_T ? 1.25
                      : amode == A_TRANSPOSED || bmode == B_TRANSPOSED ? 1.08 : 1.0;
  auto price = [&](double items, double n) {
    return 4.0 + slower * n * (items / cus * 0.33 > 0.4 ? items / cus * 0.33 : 0.4);
  };
  double cost = price(tiles, steps);
  for (int cut = 2; cut <= steps / 4 && tiles * cut <= 7.0 * cus; cut++) {
    const double c = price(tiles * cut, steps / cut) + 4.5 + 2.0 * tiles * cut * 64 * 64 * 4 / 5.0e6;
    if (c < cost) cost = c;
  }
  return cost;
}

template <class T, int AMODE, int BMODE, int BLOCKED, bool VEC>
static int launch_cfg(tfhip_ctx* ctx, GemmArgs p, const SplitPlan& pl) {
  static const char* const a_names[] = {"rowmajor", "transposed", "im2col", "im2col_up", "im2col_t", "im2col"};
  static const char* const b_names[] = {"f32", "f32t"};
  ctx->name_kernel("gemm_split_%dx%d_%s_%s%s%s", T::BM, T::BN, a_names[AMODE], b_names[BMODE],
                   VEC ? "" : "_unaligned", pl.splits > 1 ? pl.full ? "_tailk" : "_splitk" : "");
  p.tiles_m = pl.tiles_m;
  p.tiles_n = pl.tiles_n;
  p.tiles_n_shift = (pl.tiles_n & (pl.tiles_n - 1)) == 0 ? __builtin_ctz((unsigned)pl.tiles_n) : -1;
  p.col_groups = 1;
  p.cg_shift = 0;
  p.full_tiles = pl.full;
  p.tail_tiles = pl.tail;
  p.splits = pl.splits;
  p.kt_per = pl.kt_per;
  p.k_tiles = (int)ceil_div(p.K, SK);
  p.minis = 0;
  p.reverse = ctx->take_sweep();
  p.partials = nullptr;
  Temp partials(ctx);
  if (pl.splits > 1) {
    const size_t need = (size_t)pl.tail * pl.splits * T::BM * T::BN * sizeof(float);
    if (int rc = partial_tiles(ctx, need, &partials, &p.partials)) return rc;
  }
  tfhip::launch(ctx, (gemm_split_kernel<T, AMODE, BMODE, BLOCKED, VEC>),
                dim3((unsigned)(pl.full + (long long)pl.tail * pl.splits)), dim3(T::THREADS), 0, p);
  TFHIP_LAUNCH_CHECK(ctx);
  return pl.splits > 1 ? launch_splitk_finish(ctx, p, T::BM, T::BN) : TFHIP_OK;
}

template <int AMODE, int BMODE, bool KBLOCKED, bool VEC>
static int launch_mode(tfhip_ctx* ctx, const GemmArgs& p, int batch, int amode32) {
  using Big = SplitCfg<2, 2, 2>;   // 128 x 128
  using Wide = SplitCfg<2, 2, 1>;  // 64 x 128
  using Tall = SplitCfg<4, 1, 1>;  // 128 x 64
  using High = SplitCfg<4, 1, 2>;  // 256 x 64
  const int cus = ctx->num_cus, any = 0x7fffffff;
  SplitPlan pl;
  // (the registers of a 128 x 128 tile hold no third set of sums)
  // (a workgroup alone waits longer for a gather along the pixels)
  const double wait = AMODE == A_IM2COL_T ? 1.35 : 1.0;
  plan_cfg(pl, 0, Big::BM, Big::BN, 0.80 * wait, 0.80, KBLOCKED ? SPLIT_PLAIN_K / SK : any, p, batch, cus);
  plan_cfg(pl, 1, Wide::BM, Wide::BN, 0.56 * wait, 0.48, any, p, batch, cus);
  plan_cfg(pl, 2, Tall::BM, Tall::BN, 0.60 * wait, 0.58, any, p, batch, cus);
  constexpr bool HIGH = AMODE != A_IM2COL_T && AMODE != A_IM2COL;  // (one pixel position per thread; registers)
  if constexpr (HIGH)
    plan_cfg(pl, 3, High::BM, High::BN, 1.20, 0.88, KBLOCKED ? SPLIT_PLAIN_K / SK : any, p, batch, cus);
  if (pl.cfg < 0 || pl.cost > float32_cost(p, batch, cus, amode32, BMODE)) return -1;
  // tfhip_matmul_noalloc takes the same plan where its array holds the partial tiles, and float32
  // where not: the split kernels' cuts are larger than those it has always taken.
  const size_t tile = pl.cfg == 0   ? Big::BM * Big::BN
                      : pl.cfg == 1 ? Wide::BM * Wide::BN
                      : pl.cfg == 2 ? Tall::BM * Tall::BN
                                    : High::BM * High::BN;
  if (ctx->no_alloc && pl.splits > 1 && (size_t)pl.tail * pl.splits * tile * sizeof(float) > kScratchBytes) return -1;
  const int longest = pl.full ? (int)ceil_div(p.K, SK) : pl.kt_per;
  const bool blocked = KBLOCKED && longest * SK > SPLIT_PLAIN_K;
#define TFHIP_LAUNCH(T)                                                            \
  return blocked ? launch_cfg<T, AMODE, BMODE, KBLOCKED ? SPLIT_BLOCK : 0, VEC>(ctx, p, pl) \
                 : launch_cfg<T, AMODE, BMODE, 0, VEC>(ctx, p, pl)
  switch (pl.cfg) {
    case 0: return launch_cfg<Big, AMODE, BMODE, 0, VEC>(ctx, p, pl);
    case 1: TFHIP_LAUNCH(Wide);
    case 2: TFHIP_LAUNCH(Tall);
    default:
      if constexpr (HIGH) return launch_cfg<High, AMODE, BMODE, 0, VEC>(ctx, p, pl);
      else return -1;
  }
#undef TFHIP_LAUNCH
}

// Which products come here: transposed and batched ones and the gradients of convolutions, where
// the two estimates above say so.  Measured on MI355X with normal values, float32 kernels against
// these, kernel times: [3000, 1000]^T-shaped x [1000, 3000] 192 -> 165 us, [1500, 3000] x [3000, 900]^T
// 94 -> 81, 3 x [1280, 1600] x [1600, 2240] 245 -> 203, 96 x [201, 67] x [67, 201] 24.6 -> 13.2, 3 x 3 filter
// gradient of [32, 56, 56, 64] -> 128 157 -> 114, its input gradient 185 -> 116 (139 in tiles of [128, 64] and
// with the taps placed per lane), 5 x 5 of [8, 28, 28, 64] <- 256 84 -> 52.
// Small products are quicker there (16 x [128, 128] x [128, 128] 5.3 against 8.2, [1000, 256] x [256, 100] 10.4 against
// 12.5).  Row-major products of one batch entry, and with them the pointwise convolutions, and
// forward convolutions have not been moved: the float32 kernels' tile choice for them is asserted by
// name at some sizes, and the results of relu and max pooling behind a forward convolution change
// with its rounding, whichever that is.
int launch_split(tfhip_ctx* ctx, const GemmArgs& q, int batch, int amode, int bmode, bool kblocked,
                 long long a_bytes, long long b_bytes) {
  if (q.M < 1 || q.N < 1 || q.K < SPLIT_LEAST_K || batch < 1) return -1;
  if (batch == 1 && amode == A_ROWMAJOR && bmode != B_TRANSPOSED) return -1;
  if (amode == A_IM2COL) return -1;
  // 32-bit byte offsets, also of the steps past the last k and of a tile of the result
  const long long lim = 0x7fffffffLL - 64LL * 4 * (q.lda > q.ldb ? q.lda : q.ldb);
  if (a_bytes > lim || b_bytes > lim) return -1;
  if (q.N >= (1 << 22) || q.lda >= (1 << 22) || q.ldb >= (1 << 22)) return -1;
  const int amode32 = amode;
  if (amode == A_IM2COL_UP) {
    if (q.up_h != 1 || q.up_w != 1) return -1;
    amode = A_IM2COL;
  }
  const bool vec = q.a_vec && q.b_vec;
  if (amode == A_IM2COL && vec && q.Cin % SK == 0 && q.KH * q.KW < 32) amode = A_IM2COL_TAPS;
  if (bmode == B_UINT8 || (!vec && (amode == A_IM2COL || amode == A_IM2COL_T))) return -1;
  GemmArgs p = q;
  p.a_bytes = (unsigned)a_bytes;
  p.b_bytes = (unsigned)b_bytes;
  if (amode == A_IM2COL_TAPS) {
    p.by_cin = Divisor(p.Cin);
    p.by_kw = Divisor(p.KW);
  }
#define TFHIP_CASE(AM, BM_, KB, V)                               \
  if (amode == AM && bmode == BM_ && kblocked == KB && vec == V) \
    return launch_mode<AM, BM_, KB, V>(ctx, p, batch, amode32);
  TFHIP_CASE(A_ROWMAJOR, B_ROWMAJOR, true, true)
  TFHIP_CASE(A_ROWMAJOR, B_TRANSPOSED, true, true)
  TFHIP_CASE(A_TRANSPOSED, B_ROWMAJOR, true, true)
  TFHIP_CASE(A_TRANSPOSED, B_TRANSPOSED, true, true)
  TFHIP_CASE(A_ROWMAJOR, B_ROWMAJOR, true, false)
  TFHIP_CASE(A_ROWMAJOR, B_TRANSPOSED, true, false)
  TFHIP_CASE(A_TRANSPOSED, B_ROWMAJOR, true, false)
  TFHIP_CASE(A_TRANSPOSED, B_TRANSPOSED, true, false)
  TFHIP_CASE(A_IM2COL, B_ROWMAJOR, false, true)
  TFHIP_CASE(A_IM2COL_TAPS, B_ROWMAJOR, false, true)
  TFHIP_CASE(A_IM2COL_T, B_ROWMAJOR, false, true)
#undef TFHIP_CASE
  return -1;
}

}  // namespace tfhip
