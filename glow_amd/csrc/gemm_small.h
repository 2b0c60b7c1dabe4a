// The int8 contraction for outputs too small to fill the chip with 64x64 tiles:
// a FullyConnected over a small batch, every layer of an image network that
// answers one image. Such a launch is as long as its longest chain of dependent
// steps, so the work is cut fine: 32x32 output tiles, the K loop of a tile split
// over the W waves (4 or 8) of its workgroup.
//
// A wave takes every W-th 32-byte K step. Its operand fragments go from global
// memory straight into registers in the matrix-core layout (lane l feeds 16
// consecutive k-bytes of row l % 32; no LDS staging: each byte is used by one wave
// only), several steps in flight before the first multiply. The partial 32x32
// accumulators meet in LDS and 256 threads finish four neighbouring columns each:
// one 4-byte store, one 4-byte residual load that was asked for ahead of the K
// loop, the columns' constants from a table that the last wave made meanwhile (in
// every wave the ten optional parameter arrays are 200 instructions that the launch
// waits for). int32 partial sums add in any order to the same bits, so the result is
// that of the unsplit loop.
//
// What it measured against the kernels for larger problems (us, before / after):
// FullyConnected 1 x 4096 x 4096 12.7 / 7.3, 6 x 3831 x 5 21.3 / 8.4, 61 x 415 x 509
// with weight offsets 7.7 / 7.1, 1024 x 1024 x 256 6.5 / 4.2; 3x3 windows over a
// 14x14x256 image 12.5 / 7.7, 7x7x512 20.5 / 10.6, 40x40x24 36.8 / 5.8. A launch that
// does nothing takes 3 us in the same chain; the rest is the K steps of a wave, about
// 0.4 us for each group of loads it waits for.
//
// Operands: dense rows of any length and alignment, convolution windows over
// channels in fours (groups too), weight offsets and sums formed in the kernel
// (SUMS: both operands' sums as soon as one is needed, and the requantisation without
// its hints), the fused residual add.
#ifndef GLOW_MI355X_GEMM_SMALL_H
#define GLOW_MI355X_GEMM_SMALL_H

#include "gemm_i8.h"

namespace mi355x {

// How rows are read: whole 16-byte chunks on 16-byte boundaries; dense rows at any
// byte; convolution windows word by word.
enum SmallRead { kSmallChunks, kSmallBytes, kSmallWords };

// 16 bytes at any address
struct __attribute__((packed, aligned(1))) AnyChunk { int x, y, z, w; };
__device__ __forceinline__ v4i load_any16(const int8_t *p) {
  const AnyChunk c = *reinterpret_cast<const AnyChunk *>(p);
  return v4i{c.x, c.y, c.z, c.w};
}
__device__ __forceinline__ int dot_ones(v4i v, int acc) {
#pragma unroll
  for (int j = 0; j < 4; j++) acc = __builtin_amdgcn_sdot4(v[j], 0x01010101, acc, false);
  return acc;
}
// The bytes [k, k + 16) of a dense row of K bytes, zeros past its end.
__device__ __forceinline__ v4i row_end16(const int8_t *row, int k, int K) {
  if (K >= 16) {
    // the 16 bytes that end with the row, moved down
    const v4i c = load_any16(row + min(k, K - 16));
    const int n = min(max(k - (K - 16), 0), 16);
    unsigned __int128 x = ((unsigned __int128)(((uint64_t)(uint32_t)c[3] << 32) | (uint32_t)c[2]) << 64) |
                          (((uint64_t)(uint32_t)c[1] << 32) | (uint32_t)c[0]);
    x = n >= 16 ? 0 : x >> (8 * n);
    return v4i{(int)(uint32_t)x, (int)(uint32_t)(x >> 32), (int)(uint32_t)(x >> 64), (int)(uint32_t)(x >> 96)};
  }
  uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
  for (int b = 0; b < 16; b++) {
    const uint32_t v = (uint8_t)row[min(k + b, K - 1)];
    w[b >> 2] |= (k + b < K ? v : 0u) << (8 * (b & 3));
  }
  return v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
}

// Four results of one row, columns c .. c + 3 of the tile.
template <int MODE>
__device__ __forceinline__ void small_requant(int32_t (&y)[4], const v4i &sum, const int32_t *par,
                                              const Epilogue &ep) {
  const v4i colc = *reinterpret_cast<const v4i *>(par + kParColc * 32);
  const v4i pre = *reinterpret_cast<const v4i *>(par + kParPre * 32);
  const v4i scale = *reinterpret_cast<const v4i *>(par + kParScale * 32);
  const v4i post = *reinterpret_cast<const v4i *>(par + kParPost * 32);
  const v4i fold = *reinterpret_cast<const v4i *>(par + kParFold * 32);
#pragma unroll
  for (int j = 0; j < 4; j++) {
    if constexpr (MODE == 3)
      y[j] = (int32_t)((uint32_t)__mul24(sum[j], scale[j]) + (uint32_t)fold[j]) >> post[j];
    else if constexpr (MODE == 1)
      y[j] = (int32_t)((uint32_t)__mul24((int32_t)((uint32_t)sum[j] + (uint32_t)colc[j]) >> pre[j],
                                         scale[j]) +
                       (uint32_t)fold[j]) >> post[j];
    else
      y[j] = scale_i32((int32_t)((uint32_t)sum[j] + (uint32_t)colc[j]), pre[j], post[j], scale[j],
                       ep.out_off);
  }
}

template <class ARows, int W, int READ, bool SUMS>
__global__ __launch_bounds__(W * 64) void gemm_i8_small_kernel(ARows A, DenseRows B, Epilogue ep,
                                                               int M, int N, int K, int tiles_m,
                                                               int tiles_n, int by_column,
                                                               long long b_group_stride) {
  // fewer steps in flight where a wave's registers or its address arithmetic are
  // what is short
  constexpr int kChunk = W == 8 || READ == kSmallWords ? 4 : 8;
  __shared__ __attribute__((aligned(16))) int32_t s_part[W][16][64]; // [wave][register][lane]
  __shared__ __attribute__((aligned(16))) int32_t s_par[kParArrays * 32];
  __shared__ int32_t s_woff[SUMS ? 32 : 1];
  __shared__ int32_t s_sa[SUMS ? W : 1][64], s_sb[SUMS ? W : 1][64];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, lhi = lane >> 5;
  // blockIdx.x runs along the larger operand and is padded to a multiple of the
  // eight dies, over which consecutive blocks are dealt: a die then has every
  // eighth tile row of that operand to itself and its L2 holds all of the other.
  const int tm = by_column ? blockIdx.y : blockIdx.x, tn = by_column ? blockIdx.x : blockIdx.y;
  if (tm >= tiles_m || tn >= tiles_n) return;      // uniform over the block
  const int m0 = tm * 32, n0 = tn * 32;
  const int group = (int)blockIdx.z, n_base = group * N;
  A.set_group(group);

  // rows past the end re-read the last row; their results are not stored
  const auto arow = A.row(min(m0 + l32, M - 1));
  const int8_t *brow = B.p + group * b_group_stride + (long long)min(n0 + l32, N - 1) * B.ld;

  v16i acc;
#pragma unroll
  for (int r = 0; r < 16; r++) acc[r] = 0;
  int sa = 0, sb = 0;

  const int steps = K / 32;                       // whole 32-byte K steps
  v4i af[kChunk], bf[kChunk];
  auto request = [&](int base) {
#pragma unroll
    for (int u = 0; u < kChunk; u++) {
      // steps past the end re-read the last step and are not used
      const int s = min(base + W * u, steps - 1);
      if constexpr (READ == kSmallChunks) {
        af[u] = *reinterpret_cast<const v4i *>(A.step_ptr(arow, s * 32, lhi * 16));
        bf[u] = *reinterpret_cast<const v4i *>(brow + s * 32 + lhi * 16);
      } else {
        if constexpr (READ == kSmallBytes) {
          af[u] = load_any16(A.step_ptr(arow, s * 32, lhi * 16));
        } else {
          const int4 v = A.load_words(arow, s * 32 + lhi * 16, K);
          af[u] = v4i{v.x, v.y, v.z, v.w};
        }
        bf[u] = load_any16(brow + s * 32 + lhi * 16);
      }
    }
  };
  int base = wave;
  if (base < steps) request(base);
  // the row's end, K % 32 bytes: one step more of the wave whose turn it is
  const bool tail = (K & 31) != 0 && wave == steps % W;
  v4i at{0, 0, 0, 0}, bt{0, 0, 0, 0};
  if (tail) {
    const int k = steps * 32 + lhi * 16;
    if constexpr (READ == kSmallChunks) {
      if (k < K) {
        at = *reinterpret_cast<const v4i *>(A.step_ptr(arow, steps * 32, lhi * 16));
        bt = *reinterpret_cast<const v4i *>(brow + k);
      }
    } else {
      if constexpr (READ == kSmallBytes) {
        at = row_end16(A.step_ptr(arow, 0, 0), k, K);
      } else {
        const int4 v = A.load_words(arow, k, K);
        at = v4i{v.x, v.y, v.z, v.w};
      }
      bt = row_end16(brow, k, K);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // what the 256 finishing threads need of the residual
  const int row = tid >> 3, c4 = (tid & 7) * 4;    // four columns of one row
  const int m = m0 + row, n = n0 + c4;
  const bool mine = tid < 256 && m < M && n < N;
  const long long place = (long long)m * ep.ldc + n_base + n;
  const bool words = mine && n + 4 <= N && ((((uintptr_t)ep.out + place) & 3) == 0) &&
                     ((((uintptr_t)ep.add.res + place) & 3) == 0 || !ep.add.res);
  uint32_t res = 0;
  if (ep.add.res && mine) {
    if (words) {
      res = *reinterpret_cast<const uint32_t *>(ep.add.res + place);
    } else {
      for (int j = 0; j < min(4, N - n); j++)
        res |= (uint32_t)(uint8_t)ep.add.res[place + j] << (8 * j);
    }
  }
  const int mode = SUMS ? 0 : requant_mode(ep);
  if (wave == W - 1) {
    ColRaw col[1];
    load_col_raw<1, 32>(col, ep, N, n0, n_base, 0, l32);
    if (lane < 32) {
      par_table_store<32>(s_par, lane, col[0], ep, K, mode);
      if constexpr (SUMS) s_woff[lane] = col[0].woff;
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  while (base < steps) {
#pragma unroll
    for (int u = 0; u < kChunk; u++)
      if (base + W * u < steps) {
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[u], bf[u], acc, 0, 0, 0);
        if constexpr (SUMS) {
          sa = dot_ones(af[u], sa);
          sb = dot_ones(bf[u], sb);
        }
      }
    base += W * kChunk;
    if (base < steps) request(base);
  }
  if (tail) {
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(at, bt, acc, 0, 0, 0);
    if constexpr (SUMS) {
      sa = dot_ones(at, sa);
      sb = dot_ones(bt, sb);
    }
  }

  // the partial tiles meet in LDS
  if constexpr (SUMS) {
    s_sa[wave][lane] = sa;
    s_sb[wave][lane] = sb;
  }
#pragma unroll
  for (int r = 0; r < 16; r++) s_part[wave][r][lane] = acc[r];
  __syncthreads();
  if (!mine) return;

  // element (row, col) lies in register 4 (row / 8) + row % 4 of lane
  // col + 32 ((row / 4) % 2)
  const int reg = 4 * (row >> 3) + (row & 3), src = c4 + 32 * ((row >> 2) & 1);
  v4i sum{0, 0, 0, 0};
#pragma unroll
  for (int w = 0; w < W; w++) sum += *reinterpret_cast<const v4i *>(&s_part[w][reg][src]);
  if constexpr (SUMS) {
    uint32_t rs = 0;                               // of the row of A
#pragma unroll
    for (int w = 0; w < W; w++) rs += (uint32_t)s_sa[w][row] + (uint32_t)s_sa[w][row + 32];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      uint32_t x = (uint32_t)sum[j] - (uint32_t)s_woff[c4 + j] * rs;
      if (!ep.sum_b) {
        uint32_t cs = 0;                           // of the row of B
#pragma unroll
        for (int w = 0; w < W; w++) cs += (uint32_t)s_sb[w][c4 + j] + (uint32_t)s_sb[w][c4 + j + 32];
        x -= (uint32_t)ep.a_off * cs;
      }
      sum[j] = (int)x;
    }
  }
  int32_t y[4];
  const int32_t *par = s_par + c4;
  if (mode == 3) small_requant<3>(y, sum, par, ep);
  else if (mode == 1) small_requant<1>(y, sum, par, ep);
  else small_requant<0>(y, sum, par, ep);
  int32_t lo, hi;
  activation_clamp(ep, lo, hi);
#pragma unroll
  for (int j = 0; j < 4; j++) {
    if (ep.act == 5 && y[j] < ep.out_off)
      y[j] = scale_i32((int32_t)((uint32_t)y[j] - (uint32_t)ep.out_off), ep.a0, ep.a1, ep.a2,
                       ep.out_off);
    y[j] = med3_i32(y[j], lo, hi);
  }
  uint32_t word = pack4_sat8(y[0], y[1], y[2], y[3], 0);
  if (ep.add.res) word = fused_add_word(word, res, ep.add);
  else if (ep.add.relu) word = fused_relu_word(word, ep.add);
  if (words) {
    *reinterpret_cast<uint32_t *>(ep.out + place) = word;
  } else {
    for (int j = 0; j < min(4, N - n); j++) ep.out[place + j] = (int8_t)(word >> (8 * j));
  }
}

// Whether a product is small enough for this kernel: at most one 32x32 tile per
// compute unit for dense rows. With a second tile on some of them the 64x64 tiles,
// which read each operand half as often, are level or ahead (us, this kernel / those,
// M384 N768, 288 tiles: K512 6.0 / 4.5, K2048 9.3 / 8.0; M512 N512, 256 tiles: 4.3 /
// 4.5 and 6.2 / 8.0). The larger kernels spend more on a convolution window, so
// the line lies further out there (ConvRows::small_tiles). One row of tiles over long
// rows reads every weight once in either kernel, here without the other's LDS ring
// filled half with rows past M: M16 K1024 N32768 14.6 / 9.4 (the other / this), N65536
// 23.1 / 16.0, M16 K4096 N16384 19.4 / 17.5; with K415 N16384 7.6 / 10.0.
template <class ARows>
static bool small_applies(const ARows &A, const GemmShape &g, bool aligned) {
  int tiles_per_unit = A.small_tiles(aligned, g.K);
  if (tiles_per_unit == 1 && aligned && g.M <= 32 && g.K >= 1024) tiles_per_unit = 8;
  return (long long)((g.M + 31) / 32) * ((g.N + 31) / 32) * g.groups <=
         (long long)tiles_per_unit * gemm_cus();
}

template <class ARows, int W, int READ, bool SUMS>
static int gemm_small_launch_as(const ARows &A, const DenseRows &B, const Epilogue &ep,
                                const GemmShape &g, hipStream_t st) {
  const int tiles_m = (g.M + 31) / 32, tiles_n = (g.N + 31) / 32;
  const bool by_column = g.N > g.M;
  const unsigned along = (unsigned)((by_column ? tiles_n : tiles_m) + 7) / 8 * 8;
  const unsigned across = (unsigned)(by_column ? tiles_m : tiles_n);
  MI355X_REQUIRE(across < 65536 && g.groups < 65536, "problem too large");
  hipLaunchKernelGGL((gemm_i8_small_kernel<ARows, W, READ, SUMS>),
                     dim3(along, across, (unsigned)g.groups), dim3(W * 64), 0, st, A, B, ep, g.M, g.N,
                     g.K, tiles_m, tiles_n, (int)by_column, g.b_group_stride);
  return check_launch("gemm_i8_small");
}

// Eight waves per tile while two such workgroups per compute unit hold all tiles;
// four where there are more, which keeps as many bytes in flight with half the
// constants tables and partial tiles (3565 x 200 x 864 windows, 784 tiles: 8.1 us by
// four waves, 8.9 by eight; 784 x 128 x 1152, 100 tiles: 6.2 and 5.2).
template <class ARows, int READ, bool SUMS>
static int gemm_small_launch_waves(const ARows &A, const DenseRows &B, const Epilogue &ep,
                                   const GemmShape &g, hipStream_t st) {
  const long long tiles = (long long)((g.M + 31) / 32) * ((g.N + 31) / 32) * g.groups;
  if (tiles <= 2 * gemm_cus()) return gemm_small_launch_as<ARows, 8, READ, SUMS>(A, B, ep, g, st);
  return gemm_small_launch_as<ARows, 4, READ, SUMS>(A, B, ep, g, st);
}

template <class ARows>
static int gemm_small_launch(const ARows &A, const DenseRows &B, const Epilogue &ep,
                             const GemmShape &g, bool sums, bool aligned, hipStream_t st) {
  constexpr int kOther = ARows::kDense ? kSmallBytes : kSmallWords;
  if (aligned)
    return sums ? gemm_small_launch_waves<ARows, kSmallChunks, true>(A, B, ep, g, st)
                : gemm_small_launch_waves<ARows, kSmallChunks, false>(A, B, ep, g, st);
  return sums ? gemm_small_launch_waves<ARows, kOther, true>(A, B, ep, g, st)
              : gemm_small_launch_waves<ARows, kOther, false>(A, B, ep, g, st);
}

} // namespace mi355x
#endif
