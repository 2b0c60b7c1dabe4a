// The int8 contraction for outputs too small to fill the chip with 64x64 tiles:
// a FullyConnected over a small batch, every layer of an image network that
// answers one image. Such a launch is as long as its longest chain of dependent
// steps, so the work is cut fine: 16x16 or 32x32 output tiles, the K loop of a tile
// split over the four waves of its workgroup (eight where rows are read by words).
//
// A wave takes every W-th K step (64 bytes of 16 rows or 32 of 32). Its operand
// fragments go from global memory straight into registers in the matrix-core layout (a
// lane feeds 16 consecutive k-bytes of one row; no LDS staging: each byte is used by one
// wave only), six or eight steps in flight, each asked for again as soon as it is
// multiplied. The partial tiles meet in LDS and T * T / 4 threads finish four
// neighbouring columns each: one 4-byte store, one 4-byte residual load that was asked
// for ahead of the K loop, the columns' constants from a table that the last wave made
// meanwhile (in every wave the ten optional parameter arrays are 200 instructions that
// the launch waits for). int32 partial sums add in any order to the same bits, so the
// result is that of the unsplit loop.
//
// What bounds it: a launch that does nothing takes 3 us in the same chain; behind that
// the rate at which one CU pulls rows from L2, some 45 bytes per ns in pieces of 64
// bytes, which is why 16x16 tiles (four times the workgroups, half the bytes each) win
// while they still fit one or two per CU, and why no step is asked for in vain. More
// waves do not help (16x16 tiles of 8 / 16 waves on 3x3 over 14x14x256: 5.0 / 8.5 us,
// 4.9 with four). us, 32x32 tiles of eight waves with re-read steps / now: FullyConnected
// 61 x 415 x 509 with weight offsets 7.1 / 4.0, 1 x 4096 x 4096 7.5 / 5.4, 64 x 2048 x
// 1000 6.3 / 4.3, 128 x 1024 x 1024 4.5 / 4.5; 3x3 windows over 14x14x256 8.0 / 4.9,
// 7x7x512 10.9 / 6.7, 28x28x128 5.5 / 4.8; pointwise 14x14, 256 to 1024 4.5 / 3.4, 7x7,
// 2048 to 512 6.2 / 4.1.
//
// Operands: dense rows of any length and alignment, convolution windows over
// channels in fours (groups too), weight offsets and sums formed in the kernel
// (SUMS: both operands' sums as soon as one is needed, and the requantisation without
// its hints), the fused residual add.
#ifndef GLOW_MI355X_GEMM_SMALL_H
#define GLOW_MI355X_GEMM_SMALL_H

#include "gemm_i8.h"

#include <type_traits>

namespace mi355x {

// How rows are read: whole 16-byte chunks on 16-byte boundaries; dense rows by loads of
// sixteen bytes wherever they start (on a word, or few enough bytes: shift_bytes); dense rows
// at any byte by words; convolution windows word by word.
enum SmallRead { kSmallChunks, kSmallQuads, kSmallBytes, kSmallWords };

__device__ __forceinline__ v4i load_any16(const int8_t *p) {
  const AnyChunk c = *reinterpret_cast<const AnyChunk *>(p);
  return v4i{c.x, c.y, c.z, c.w};
}
// Sixteen bytes from any address as the four words that hold them from the first on and a
// fifth: a sixteen-byte load that does not start on a word takes three times as long as one
// that does (FullyConnected 300 x 4004 x 300 7.6 us, 300 x 4001 x 300 21.7; 12.4 with this). Every word read
// holds a byte that is asked for, or is read twice, so that none lies past the memory of the
// rows by more than the rest of a word.
struct Shifted {
  v4i lo;
  int hi;
};
__device__ __forceinline__ Shifted load_shifted(const int8_t *words, int shift) {
  struct __attribute__((packed, aligned(4))) Quad { int x, y, z, w; };
  const Quad q = *reinterpret_cast<const Quad *>(words);
  return Shifted{v4i{q.x, q.y, q.z, q.w}, *reinterpret_cast<const int *>(words + (shift ? 16 : 12))};
}
__device__ __forceinline__ v4i unshift(const Shifted &s, int shift) {
  return v4i{(int)__builtin_amdgcn_alignbyte(s.lo[1], s.lo[0], shift),
             (int)__builtin_amdgcn_alignbyte(s.lo[2], s.lo[1], shift),
             (int)__builtin_amdgcn_alignbyte(s.lo[3], s.lo[2], shift),
             (int)__builtin_amdgcn_alignbyte(s.hi, s.lo[3], shift)};
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

// The matrix-core instruction of a T x T tile: its K step in bytes, the registers a lane
// holds of the result, and where element (row, col) of the tile lies in them.
template <int T> struct SmallTile;
template <> struct SmallTile<32> {
  static constexpr int kStep = 32, kRegs = 16;
  typedef v16i Acc;
  static __device__ __forceinline__ Acc mfma(v4i a, v4i b, Acc c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int reg(int row) { return 4 * (row >> 3) + (row & 3); }
  static __device__ __forceinline__ int lane(int row, int col) { return col + 32 * ((row >> 2) & 1); }
};
template <> struct SmallTile<16> {
  static constexpr int kStep = 64, kRegs = 4;
  typedef v4i Acc;
  static __device__ __forceinline__ Acc mfma(v4i a, v4i b, Acc c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int reg(int row) { return row & 3; }
  static __device__ __forceinline__ int lane(int row, int col) { return col + 16 * (row >> 2); }
};

// Four results of one row, columns c .. c + 3 of the tile.
template <int MODE, int T>
__device__ __forceinline__ void small_requant(int32_t (&y)[4], const v4i &sum, const int32_t *par,
                                              const Epilogue &ep) {
  const v4i colc = *reinterpret_cast<const v4i *>(par + kParColc * T);
  const v4i pre = *reinterpret_cast<const v4i *>(par + kParPre * T);
  const v4i scale = *reinterpret_cast<const v4i *>(par + kParScale * T);
  const v4i post = *reinterpret_cast<const v4i *>(par + kParPost * T);
  const v4i fold = *reinterpret_cast<const v4i *>(par + kParFold * T);
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

template <class ARows, int T, int W, int READ, bool SUMS>
__global__ __launch_bounds__(W * 64, 4) void gemm_i8_small_kernel(ARows A, DenseRows B, Epilogue ep,
                                                               int M, int N, int K, int tiles_m,
                                                               int tiles_n, int by_column,
                                                               long long b_group_stride) {
  typedef SmallTile<T> Tile;
  constexpr int kStep = Tile::kStep, kRegs = Tile::kRegs;
  // steps in flight: fewer where the address arithmetic is what a wave waits for, and where
  // more would not fit the 128 registers of four waves per SIMD (a spill, and be it of two
  // registers, makes the launch 1 us longer: M1099 K15 N122 4.2 / 5.9 us)
  constexpr int kAhead = T == 16 || READ == kSmallBytes ? 6 : READ == kSmallWords ? 4 : SUMS ? 7 : 8;
  __shared__ __attribute__((aligned(16))) int32_t s_part[W][kRegs][64]; // [wave][register][lane]
  __shared__ __attribute__((aligned(16))) int32_t s_par[kParArrays * T];
  __shared__ int32_t s_woff[SUMS ? T : 1];
  __shared__ int32_t s_sa[SUMS ? W : 1][64], s_sb[SUMS ? W : 1][64];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane % T, part = lane / T;      // the row a lane feeds, which 16 bytes of a step
  // blockIdx.x runs along the larger operand and is padded to a multiple of the
  // eight dies, over which consecutive blocks are dealt: a die then has every
  // eighth tile row of that operand to itself and its L2 holds all of the other.
  const int tm = by_column ? blockIdx.y : blockIdx.x, tn = by_column ? blockIdx.x : blockIdx.y;
  if (tm >= tiles_m || tn >= tiles_n) return;      // uniform over the block
  const int m0 = tm * T, n0 = tn * T;
  const int group = (int)blockIdx.z, n_base = group * N;
  A.set_group(group);

  // rows past the end re-read the last row; their results are not stored
  const auto arow = A.row(min(m0 + lrow, M - 1));
  const int8_t *brow = B.p + group * b_group_stride + (long long)min(n0 + lrow, N - 1) * B.ld;

  typename Tile::Acc acc;
#pragma unroll
  for (int r = 0; r < kRegs; r++) acc[r] = 0;
  int sa = 0, sb = 0;

  const int steps = K / kStep;                     // whole K steps
  // rows at any byte: how far into a word a lane's rows start, the same at every step
  constexpr bool kShift = READ == kSmallBytes;
  typedef typename std::conditional<kShift, Shifted, v4i>::type Frag;
  int a_shift = 0, b_shift = 0;
  const int8_t *a_words = nullptr, *b_words = nullptr;
  if constexpr (kShift) {
    const int8_t *a0 = A.template step_ptr<kStep>(arow, 0, part * 16), *b0 = brow + part * 16;
    a_shift = (int)((uintptr_t)a0 & 3);
    b_shift = (int)((uintptr_t)b0 & 3);
    a_words = a0 - a_shift;
    b_words = b0 - b_shift;
  }
  Frag af[kAhead], bf[kAhead];
  auto request = [&](int u, int s) {
    if constexpr (kShift) {
      af[u] = load_shifted(a_words + s * kStep, a_shift);
      bf[u] = load_shifted(b_words + s * kStep, b_shift);
    } else if constexpr (READ == kSmallChunks) {
      af[u] = *reinterpret_cast<const v4i *>(A.template step_ptr<kStep>(arow, s * kStep, part * 16));
      bf[u] = *reinterpret_cast<const v4i *>(brow + s * kStep + part * 16);
    } else {
      if constexpr (READ == kSmallQuads) {
        af[u] = load_any16(A.template step_ptr<kStep>(arow, s * kStep, part * 16));
      } else {
        const int4 v = A.load_words(arow, s * kStep + part * 16, K);
        af[u] = v4i{v.x, v.y, v.z, v.w};
      }
      bf[u] = load_any16(brow + s * kStep + part * 16);
    }
  };
  auto multiply_whole = [&](const v4i &a, const v4i &b) {
    acc = Tile::mfma(a, b, acc);
    if constexpr (SUMS) {
      sa = dot_ones(a, sa);
      sb = dot_ones(b, sb);
      // (here and now: left to itself the compiler forms the sums of conditional steps
      // ahead of their conditions and keeps them all, 184 registers or spills)
      asm volatile("" : "+v"(sa), "+v"(sb));
    }
  };
  auto multiply = [&](const Frag &a, const Frag &b) {
    if constexpr (kShift) {
      multiply_whole(unshift(a, a_shift), unshift(b, b_shift));
      __builtin_amdgcn_sched_barrier(0);           // (not the shifts of several steps at once)
    } else {
      multiply_whole(a, b);
    }
  };
  // A wave's steps are wave, wave + W, ... . Only steps that exist are asked for: a
  // load that re-reads the last one costs as much of the CU's path to L2 as one that is
  // used (3x3 over 14x14x256, 9 steps a wave in rounds of 4: 8.0 us with them, 6.8
  // without). The branches are uniform; a full round has none, so that its waits count
  // the loads exactly.
  int todo = (steps - wave + W - 1) / W, base = wave;
  if (todo >= kAhead) {
#pragma unroll
    for (int u = 0; u < kAhead; u++) request(u, base + W * u);
  } else {
#pragma unroll
    for (int u = 0; u < kAhead; u++)
      if (u < todo) request(u, base + W * u);
  }
  // the row's end, K % kStep bytes: one step more of the wave whose turn it is
  const bool tail = K % kStep != 0 && wave == steps % W;
  v4i at{0, 0, 0, 0}, bt{0, 0, 0, 0};
  if (tail) {
    const int k = steps * kStep + part * 16;
    if constexpr (READ == kSmallChunks) {
      if (k < K) {
        at = *reinterpret_cast<const v4i *>(A.template step_ptr<kStep>(arow, steps * kStep, part * 16));
        bt = *reinterpret_cast<const v4i *>(brow + k);
      }
    } else {
      if constexpr (READ == kSmallQuads || kShift) {
        at = row_end16(A.template step_ptr<kStep>(arow, 0, 0), k, K);
      } else {
        const int4 v = A.load_words(arow, k, K);
        at = v4i{v.x, v.y, v.z, v.w};
      }
      bt = row_end16(brow, k, K);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // what the finishing threads need of the residual
  constexpr int kQuads = T / 4;
  const int row = tid / kQuads, c4 = (tid % kQuads) * 4;    // four columns of one row
  const int m = m0 + row, n = n0 + c4;
  const bool mine = tid < T * kQuads && m < M && n < N;
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
    load_col_raw<1, T>(col, ep, N, n0, n_base, 0, lrow);
    if (lane < T) {
      par_table_store<T>(s_par, lane, col[0], ep, K, mode);
      if constexpr (SUMS) s_woff[lane] = col[0].woff;
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // a step's registers are asked for again as soon as it is multiplied
  while (todo >= 2 * kAhead) {
    base += W * kAhead;
    todo -= kAhead;
#pragma unroll
    for (int u = 0; u < kAhead; u++) {
      multiply(af[u], bf[u]);
      request(u, base + W * u);
    }
  }
  if (todo >= kAhead) {
    base += W * kAhead;
    todo -= kAhead;
#pragma unroll
    for (int u = 0; u < kAhead; u++) {
      multiply(af[u], bf[u]);
      if (u < todo) request(u, base + W * u);
    }
  }
#pragma unroll
  for (int u = 0; u < kAhead; u++)
    if (u < todo) multiply(af[u], bf[u]);
  if (tail) multiply_whole(at, bt);

  // the partial tiles meet in LDS
  if constexpr (SUMS) {
    s_sa[wave][lane] = sa;
    s_sb[wave][lane] = sb;
  }
#pragma unroll
  for (int r = 0; r < kRegs; r++) s_part[wave][r][lane] = acc[r];
  __syncthreads();
  if (!mine) return;

  const int reg = Tile::reg(row), src = Tile::lane(row, c4);
  v4i sum{0, 0, 0, 0};
#pragma unroll
  for (int w = 0; w < W; w++) sum += *reinterpret_cast<const v4i *>(&s_part[w][reg][src]);
  if constexpr (SUMS) {
    uint32_t rs = 0;                               // of the row of A
#pragma unroll
    for (int w = 0; w < W; w++)
#pragma unroll
      for (int p = 0; p < 64 / T; p++) rs += (uint32_t)s_sa[w][row + T * p];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      uint32_t x = (uint32_t)sum[j] - (uint32_t)s_woff[c4 + j] * rs;
      if (!ep.sum_b) {
        uint32_t cs = 0;                           // of the row of B
#pragma unroll
        for (int w = 0; w < W; w++)
#pragma unroll
          for (int p = 0; p < 64 / T; p++) cs += (uint32_t)s_sb[w][c4 + j + T * p];
        x -= (uint32_t)ep.a_off * cs;
      }
      sum[j] = (int)x;
    }
  }
  int32_t y[4];
  const int32_t *par = s_par + c4;
  if (mode == 3) small_requant<3, T>(y, sum, par, ep);
  else if (mode == 1) small_requant<1, T>(y, sum, par, ep);
  else small_requant<0, T>(y, sum, par, ep);
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

// Whether a product is small enough for this kernel, by its number of 32x32 tiles per
// compute unit (DenseRows::small_tiles, ConvRows::small_tiles: the lines between it and
// the tiled kernels, which read each operand half as often or less). One row of tiles
// over long rows reads every weight once in either kernel, here without the other's LDS
// ring filled half with rows past M: M16 K1024 N32768 14.6 / 9.4 (the other / this),
// N65536 23.1 / 16.0, M16 K4096 N16384 19.4 / 17.5; with K415 N16384 7.6 / 10.0.
template <class ARows>
static bool small_applies(const ARows &A, const GemmShape &g, bool aligned, bool sums) {
  int tiles_per_unit = A.small_tiles(aligned, g.K, sums);
  if (ARows::kDense && aligned && g.M <= 32 && g.K >= 1024) tiles_per_unit = 8;
  return (long long)((g.M + 31) / 32) * ((g.N + 31) / 32) * g.groups <=
         (long long)tiles_per_unit * gemm_cus();
}

template <class ARows, int T, int W, int READ, bool SUMS>
static int gemm_small_launch_as(const ARows &A, const DenseRows &B, const Epilogue &ep,
                                const GemmShape &g, hipStream_t st) {
  const int tiles_m = (g.M + T - 1) / T, tiles_n = (g.N + T - 1) / T;
  const bool by_column = g.N > g.M;
  const unsigned along = (unsigned)((by_column ? tiles_n : tiles_m) + 7) / 8 * 8;
  const unsigned across = (unsigned)(by_column ? tiles_m : tiles_n);
  MI355X_REQUIRE(across < 65536 && g.groups < 65536, "problem too large");
  hipLaunchKernelGGL((gemm_i8_small_kernel<ARows, T, W, READ, SUMS>),
                     dim3(along, across, (unsigned)g.groups), dim3(W * 64), 0, st, A, B, ep, g.M, g.N,
                     g.K, tiles_m, tiles_n, (int)by_column, g.b_group_stride);
  return check_launch("gemm_i8_small");
}

// 16x16 tiles while there are at most 1.6 of them per compute unit, or 4 of a single
// column of tiles, of which 32x32 tiles would leave half empty. us, 16x16 / 32x32:
// 3x3 over 7x7x512, 1 image (128 tiles) 6.8 / 10.2, 4 (416) 10.4 / 10.5, 8 (800) 17.2 /
// 10.9; over 28x28x128, 1 image (392) 4.7 / 5.0, 2 (784) 6.7 / 5.1; 64 x 2048 x 1000
// (252) 4.3 / 6.1; 5x5 over 18x18x64 to 16 channels, 8 images (162) 3.8 / 4.3, 32 (648)
// 5.0 / 5.5. Four waves to a 32x32 tile: level with eight up to a tile per compute unit,
// ahead beyond (3x3 over 56x56x64, 4 images, 392 tiles, 5.4 / 7.2), except where rows are
// read by words, whose address arithmetic eight waves share (40x40x24, 50 tiles 4.0 /
// 4.6, 400 tiles 4.9 / 5.1, 800 tiles 8.5 / 8.9 the other way round).
static long long small_tile_count(const GemmShape &g, int T) {
  return (long long)((g.M + T - 1) / T) * ((g.N + T - 1) / T) * g.groups;
}
static bool small_tiles_of_16(const GemmShape &g) {
  const long long cus = gemm_cus(), fine = small_tile_count(g, 16);
  return 5 * fine <= 8 * cus || (g.N <= 16 && fine <= 4 * cus);
}

template <class ARows, int READ, bool SUMS>
static int gemm_small_launch_tiles(const ARows &A, const DenseRows &B, const Epilogue &ep,
                                   const GemmShape &g, hipStream_t st) {
  if (small_tiles_of_16(g))
    return gemm_small_launch_as<ARows, 16, 4, READ, SUMS>(A, B, ep, g, st);
  if constexpr (READ == kSmallWords) {
    if (small_tile_count(g, 32) <= 2LL * gemm_cus()) return gemm_small_launch_as<ARows, 32, 8, READ, SUMS>(A, B, ep, g, st);
  }
  return gemm_small_launch_as<ARows, 32, 4, READ, SUMS>(A, B, ep, g, st);
}

// Whether dense rows at any byte are long enough that words and a byte shift pay: five words
// and the shift are more instructions in front of the first product, and a load that starts
// off a word only counts where loads are what a compute unit waits for. Shorter rows take
// loads of sixteen bytes. us, those / words and shift: 16x16 tiles, one per unit or fewer,
// 61 x 333 x 509 with sums 4.05 / 4.27, 61 x 531 x 509 4.33 / 4.41, 61 x 777 x 509 4.80 / 4.52,
// more of them 300 x 195 x 300 4.33 / 4.45, 300 x 251 x 300 4.61 / 4.41; 32x32 tiles, one per unit
// 400 x 290 x 450 4.55 / 4.69, 400 x 379 x 450 5.66 / 5.25, more of them 600 x 101 x 600 4.48 / 4.56,
// 600 x 123 x 600 5.01 / 4.71, at an even length 600 x 150 x 600 4.54 / 4.64. Rows a few bytes off a
// multiple of 128 meet in the same channels of L2, where a load's second line is waited for:
// 61 x 257 x 509 4.11 / 3.93, 61 x 385 x 509 4.52 / 4.00, 61 x 511 x 509 5.31 / 4.60, but 61 x 275 x
// 509 4.02 / 4.05, 61 x 131 x 509 4.03 / 4.12.
static bool shift_bytes(const GemmShape &g) {
  if (g.K >= 250 && (g.K + 5) % 128 <= 10) return true;
  const bool fine = small_tiles_of_16(g), one = small_tile_count(g, fine ? 16 : 32) <= gemm_cus();
  return g.K >= (fine ? (one ? 640 : 240) : one ? 350 : g.K % 2 ? 120 : 180);
}

template <class ARows>
static int gemm_small_launch(const ARows &A, const DenseRows &B, const Epilogue &ep,
                             const GemmShape &g, bool sums, bool aligned, hipStream_t st) {
  constexpr int kOther = ARows::kDense ? kSmallQuads : kSmallWords;
  if constexpr (ARows::kDense) {
    // (groups are convolutions', which come by words)
    if (!aligned && (((uintptr_t)A.p | (uintptr_t)B.p | (uintptr_t)A.ld | (uintptr_t)B.ld) & 3) != 0 &&
        shift_bytes(g))
      return sums ? gemm_small_launch_tiles<ARows, kSmallBytes, true>(A, B, ep, g, st)
                  : gemm_small_launch_tiles<ARows, kSmallBytes, false>(A, B, ep, g, st);
  }
  if (aligned)
    return sums ? gemm_small_launch_tiles<ARows, kSmallChunks, true>(A, B, ep, g, st)
                : gemm_small_launch_tiles<ARows, kSmallChunks, false>(A, B, ep, g, st);
  return sums ? gemm_small_launch_tiles<ARows, kOther, true>(A, B, ep, g, st)
              : gemm_small_launch_tiles<ARows, kOther, false>(A, B, ep, g, st);
}

} // namespace mi355x
#endif
