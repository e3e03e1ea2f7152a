// What the product kernels (gemm.hip, gemm_split.hip) share: the arguments of a product and the
// order in which workgroups take its tiles.
#pragma once
#include "tfhip_internal.h"
#include "tfhip_device.h"

namespace tfhip {

// A_IM2COL_UP: the gather of conv2dDerInput (rows are input pixels, k is (filter row, filter
// column, output channel) of the flipped filter; the image gathered from is dy, stretched by
// the forward stride).  A_IM2COL_T: the gather of conv2dDerFilter (rows are (filter row,
// filter column, input channel), k runs over the output pixels (n, oh, ow)).  A_IM2COL_TAPS: A_IM2COL
// where the channels of a filter tap are whole k steps, and the taps are fewer than 32.
enum { A_ROWMAJOR = 0, A_TRANSPOSED = 1, A_IM2COL = 2, A_IM2COL_UP = 3, A_IM2COL_T = 4, A_IM2COL_TAPS = 5 };
enum { B_ROWMAJOR = 0, B_TRANSPOSED = 1, B_UINT8 = 2 };

struct GemmArgs {
  const float* A;
  const void* B;
  float* C;
  const float* bias;
  const float* prelu;
  int M, N, K;
  int lda, ldb;
  long long strideA, strideB, strideC;  // per-batch element strides
  int bias_kind, prelu_kind, act;
  int a_vec, b_vec;  // operands allow aligned 4-element accesses
  // implicit-GEMM geometry (A_IM2COL): rows are (n, oh, ow), k is (kh, kw, c)
  int H, W, Cin, OH, OW, KH, KW, sh, sw, dh, dw, pt, pl;
  Divisor by_cin, by_kw;  // A_IM2COL_TAPS
  int up_h, up_w;  // A_IM2COL_UP: forward strides (dy is read at row / up_h when divisible)
  double qscale, qmin;
  // schedule (see work_item)
  int tiles_m, tiles_n, k_tiles, full_tiles, tail_tiles, splits, kt_per;
  int tiles_n_shift;  // log2(tiles_n) when that is a power of two, else -1 (a division on the vector ALU)
  // col_groups > 1 (unbatched products without a split along K): the tiles are numbered column
  // group by column group, a group being 1 << cg_shift tile columns of every tile row, so that an
  // XCD's run of tiles lies inside one group: its L2 then reads 1 / col_groups of B and
  // col_groups / 8 of A instead of all of B and an eighth of A (see choose_col_groups).
  int col_groups, cg_shift;
  float* partials;  // [tail_tiles * splits][BM * BN] partial tiles when splits > 1
  // minis > 0: the tail tiles are not split along K over workgroups but cut into `minis` tiles
  // of 16 x 16 each, one per workgroup, whose wavefronts take mini_k_per of K each (kwaves_tile)
  int minis, mini_k_per;
  unsigned a_bytes, b_bytes;  // per-batch byte extents of A and B (buffer-load range check)
  int reverse;  // walk the tiles / row blocks of every XCD's run from the end
};

// The work of one workgroup: a whole output tile, or (when tiles are split along K to fill
// the machine) the k range [kt0, kt1) of one, written to a partial slot.
struct WorkItem {
  int tile;     // linear tile index over (batch, tile row, tile column); -1 = none
  int kt0, kt1;
  int slot;     // partial slot, -1 = finish the tile here
};

// Schedule: the first `full_tiles` workgroups take one whole tile each (ids remapped per
// XCD); the remaining tail_tiles * splits workgroups take k range h % splits of tail tile
// h / splits.  The tail workgroups are dispatched last and in hardware order, so the short
// items spread over all XCDs and CUs.
__device__ __forceinline__ WorkItem work_item(const GemmArgs& p, int block) {
  WorkItem w = {-1, 0, 0, -1};
  if (block < p.full_tiles) {
    w.tile = xcd_remap_dir(block, p.full_tiles, p.reverse);
    w.kt1 = p.k_tiles;
  } else if (block - p.full_tiles < p.tail_tiles * p.splits) {
    const int h = block - p.full_tiles;
    w.tile = p.full_tiles + h / p.splits;
    const int s = h % p.splits;
    w.kt0 = s * p.kt_per;
    w.kt1 = min(p.k_tiles, w.kt0 + p.kt_per);
    if (p.splits > 1) w.slot = h;
  }
  return w;
}

// Tile row and tile column of tile t of an unbatched product (t counts row by row, or column
// group by column group).  t is the same for the whole workgroup.
__device__ __forceinline__ void tile_row_col(const GemmArgs& p, int t, int& tm, int& tn) {
  if (p.col_groups > 1) {
    const int per = p.tiles_m << p.cg_shift;  // tiles of a column group
    int g = 0;
    while (t >= per) {  // (at most col_groups - 1 times)
      t -= per;
      g++;
    }
    tm = t >> p.cg_shift;
    tn = (g << p.cg_shift) + (t - (tm << p.cg_shift));
  } else {
    tm = p.tiles_n_shift >= 0 ? t >> p.tiles_n_shift : t / p.tiles_n;
    tn = t - tm * p.tiles_n;
  }
}

// gemm.hip: memory for the partial tiles of a product cut along K: a pool block that `block` holds,
// or (tfhip_matmul_noalloc) the static array of kScratchBytes.
constexpr size_t kScratchBytes = 8u << 20;
int partial_tiles(tfhip_ctx* ctx, size_t need, Temp* block, float** out);

// gemm.hip: adds the partial tiles [tail_tiles * splits][bm * bn] of a product cut along K.
int launch_splitk_finish(tfhip_ctx* ctx, const GemmArgs& p, int bm, int bn);

// gemm_split.hip: the product on the bf16 matrix cores, every operand as the exact sum of three
// bf16 values.  Returns -1 when the kernels for float32 operands are the better choice.
int launch_split(tfhip_ctx* ctx, const GemmArgs& p, int batch, int amode, int bmode, bool kblocked,
                 long long a_bytes, long long b_bytes);

}  // namespace tfhip
