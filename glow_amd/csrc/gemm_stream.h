// Which products the streaming kernel (gemm_stream.hip) takes, and its launch: the int8
// contraction for short K and many rows, pointwise convolutions of an image network's early
// stages and FullyConnected layers over 32, 64, 96, 128 or 256 inputs.
#ifndef GLOW_MI355X_GEMM_STREAM_H
#define GLOW_MI355X_GEMM_STREAM_H

#include "gemm_i8.h"

namespace mi355x {

constexpr int kStreamBN = 128;      // most columns of a slice

// Rows of A: dense (row m at in + m * ld), or the window a convolution without
// padding and dilation reads for output pixel m of an [N, OH, OW] grid: it
// starts at input pixel (n, oh * sH, ow * sW) of an [N, IH, IW, IC] tensor and
// has KH segments of KW * IC contiguous bytes, one input row apart (a pointwise
// convolution: one segment of IC bytes).
struct StreamRows {
  const int8_t *in;
  long long ld;
  int dense;
  int OW, OHW, IH, IW, IC, sH, sW;
  int seg_chunks;        // 32-byte chunks per segment (a power of two; K / 32: one segment)
  long long seg_stride;  // bytes between segments
  __device__ __forceinline__ const int8_t *row(int m) const {
    if (dense) return in + (long long)m * ld;
    const int n = m / OHW, r = m - n * OHW;
    const int oh = r / OW, ow = r - oh * OW;
    return in + (((long long)n * IH + (long long)oh * sH) * IW + (long long)ow * sW) * IC;
  }
  // byte offset of chunk ks of a row from the row's start
  __device__ __forceinline__ long long chunk(int ks) const {
    return (long long)(ks / seg_chunks) * seg_stride + (ks % seg_chunks) * 32;
  }
};

// Whether the streaming kernel can run this product at all: K of 64, 128 or 256 (of 32 or 96
// by the shape rule only: tile 8 refuses those), 16-byte aligned operands and output, whole
// 32-column tiles, weight offsets all zero with their row sums precomputed (no in-kernel row
// sums).
static bool stream_can_run(int M, int N, int K, bool need_sa, bool need_sb, bool aligned,
                           const Epilogue &ep) {
  if (need_sa || need_sb || !aligned) return false;
  if (K != 64 && K != 128 && K != 256 && (g_tile_override == 8 || (K != 32 && K != 96))) return false;
  // whole 32-column tiles, and whole 128-column groups once there are more than 128
  if (N % 32 != 0 || (N > kStreamBN && N % kStreamBN != 0) || M < 1) return false;
  if (ep.ldc % 16 != 0 || (((((uintptr_t)ep.out) | ((uintptr_t)ep.add.res)) & 15) != 0))
    return false;
  return true;
}

// Whether it is the default for such a product: each workgroup reads its slice of the weights
// before its first tile, so the rows or results have to be many. `apart`: the rows do not lie
// on end (a stride), which costs the tiled kernels more. K of 64, 128 and 256 from where it is no
// slower than the tile that would be chosen, by columns, over M 4096 to 300 000 and N 32 to 512
// with and without a residual (us, tiled / this: K256 N128 M8192 4.9 / 8.0, M30016 6.4 / 8.5,
// M150016 19.4 / 18.5, N512 M8192 6.5 / 8.7; K128 N128 M8192 4.6 / 6.2, M150016 16.1 / 13.7, N256
// M12544 5.8 / 6.6; K64 N512 M4096 4.9 / 5.5, M12544 7.5 / 7.1).
// K of 32 and 96, with more to gain (the tiled kernels multiply whole steps of 64 and wait
// longer on them than the product takes), from 5 x 2^19 results or 49 152 rows on; us,
// tiled / this: M180000 K96 N512 60 / 34, K32 N512 57 / 30, M320625 K96 N512 103 / 55,
// M50176 K96 N64 6.1 / 5.3, N512 with the residual 28 / 21.7, M50176 K32 N32 5.4 / 4.0,
// M5184 K32 N512 5.7 / 5.2, K96 6.0 / 5.5; below the line M12800 K96 N128 4.9 / 5.4, with
// the residual 5.2 / 6.4, M4096 K96 N512 5.4 / 5.5.
// Windows over several pixels, whose taps the tiled kernels have to locate, from 4096 on,
// those of 256 bytes with more than 64 columns from three 32x32 tiles per compute unit on (4x4
// over 16 channels, M10240 N32 5.7 / 4.4, N64 6.5 / 5.2, with the residual 7.3 / 5.9, M6784 N96
// 6.5 / 6.4, with it 7.3 / 7.7, M5120 N128 6.5 / 7.1).
static bool stream_applies(int M, int N, int K, bool window, bool apart) {
  if (M < 4096 || N > 512) return false;
  const long long results = (long long)M * N;
  if (K == 32 || K == 96) return M >= 49152 || results >= (5 << 19);
  if (window)
    return K != 256 || N <= 64 ||
           (long long)((M + 31) / 32) * ((N + 31) / 32) > 3LL * gemm_cus();
  // rows for up to 64 and up to 128 columns, results beyond
  struct Line { int rows64, rows128, results; };
  constexpr Line kLines[2][3] = {
      {{28000, 28000, 4700000}, {80000, 60000, 10000000}, {90000, 60000, 16500000}},
      {{25000, 25000, 4000000}, {40000, 40000, 4500000}, {28000, 45000, 18000000}}};
  const Line &l = kLines[apart][K == 64 ? 0 : K == 128 ? 1 : 2];
  return N <= 64 ? M >= l.rows64 : N <= 128 ? M >= l.rows128 : results >= l.results;
}

// What the rules let through (gemm_stream.hip: its kernels are built once for the library).
int gemm_stream_launch(const StreamRows &A, const int8_t *W, const Epilogue &ep, int M, int N, int K,
                       hipStream_t st);

} // namespace mi355x
#endif
