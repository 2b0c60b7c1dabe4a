// The int8 contraction for short K and many rows: pointwise convolutions of an
// image network's early stages and FullyConnected layers over 32, 64, 96, 128 or 256
// inputs, where a launch is all memory traffic and requantisation and the
// tiled kernels of gemm_i8.h spend their time in load latency, barriers and
// output staging.
//
//   * the weights of a workgroup's column slice (128 columns, at most 35 KB)
//     and the columns' requantisation constants are put in LDS once; from then
//     on the workgroup's waves never meet again;
//   * a wave walks over tiles of 32 rows: a lane loads its row's K bytes
//     straight from global memory into registers in the matrix-core layout
//     (every byte of A is read by exactly one lane), multiplies them with the
//     weight fragments read from LDS, 32 columns at a time, and requantises and
//     packs sixteen output bytes per lane (the transposed-accumulator epilogue
//     of gemm_i8.h); the slice's columns go through a wave-private
//     transpose in LDS so that they are written as whole 128-byte lines, with
//     the fused residual add read the same way;
//   * a wave asks for its next tile's rows before it works on the current one,
//     and for the next tile's residual bytes as soon as it has used the current
//     ones, so that neither is waited for (up to K = 128; at K = 256 the rows alone
//     are 32 registers a lane and the loop stays plain); three to five workgroups
//     per CU cover what is left (stream_per_cu).
// What bounds it is latency that more waves cover, then memory: at 64 x 56x56 x 64 -> 256
// 3.6 TB/s with a residual (265 vector instructions per 32x32 results of a wave), without
// one 3.3 (132). Hence the accumulators that start from the column constants, the packing
// shift (requant.h), the residual asked for a tile ahead (41.4 -> 38.9 us there) and added
// in words (-> 36.2; gemm_i8.h: fused_word_fast), and a kernel per variant, whose fewer
// registers let five workgroups share a CU (-> 32; 20.9 -> 19.9 without a residual). What
// gave nothing: 16 instructions less (a clamp that is int8's own range left to the packing),
// half the reads from LDS (two row tiles per wave sharing weights and constants: level at
// K = 64, up to twice as long at K = 256, whose waves got fewer).
//
// Results are bit for bit those of the tiled kernels (same integer sums, same
// requantisation).
#include "gemm_stream.h"

namespace mi355x {

constexpr int kStreamParBytes = kParArrays * kStreamBN * 4;

// Bytes between the rows of a wave's staging tile, by the passes of its copy-out: up to
// 128 or 64 output columns plus 16 (consecutive rows start 36 or 20 banks apart).
constexpr int stream_stage_stride(int np) { return (np == 4 ? 128 : 64) + 16; }

// The results leave through a wave-private transpose in LDS: the slice's columns
// are staged, then read back with columns / 16 lanes per row, so that
// a store instruction writes whole lines and the residual is read the same way.
// NP: passes of the copy-out (four for slices of 96 and 128 columns, two for
// narrower ones); RES: a residual is added. Both are template parameters so
// that every load has exactly one place that uses it, on every path: the
// compiler then waits for a load where it is used and nowhere else.
// A lane's share of the rows of tile t: KS pieces of 16 bytes in the
// matrix-core layout (rows past the end re-read the last row; their results are
// not stored).
template <int KS>
__device__ __forceinline__ void stream_load_rows(const StreamRows &A, v4i (&dst)[KS], int t, int M,
                                                 int lane) {
  const int8_t *ar = A.row(min(t * 32 + (lane & 31), M - 1)) + (lane >> 5) * 16;
  if (A.seg_chunks >= KS) {
#pragma unroll
    for (int ks = 0; ks < KS; ks++) dst[ks] = *reinterpret_cast<const v4i *>(ar + ks * 32);
  } else {
#pragma unroll
    for (int ks = 0; ks < KS; ks++) dst[ks] = *reinterpret_cast<const v4i *>(ar + A.chunk(ks));
  }
}

// A lane's accumulators belong to sixteen columns: they start from the columns'
// constants instead of having them added later (which modes other than 3 do).
template <int MODE> __device__ __forceinline__ v16i stream_acc_start(const int32_t *par) {
  v16i acc;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    v4i c{0, 0, 0, 0};
    if constexpr (MODE != 3) c = *reinterpret_cast<const v4i *>(par + kParColc * kStreamBN + 4 * q);
#pragma unroll
    for (int i = 0; i < 4; i++) acc[4 * q + i] = c[i];
  }
  return acc;
}

// af: the rows of the wave's first tile, asked for by the caller.
template <int KS, int NP, bool RES, int MODE, bool LEAKY>
__device__ __forceinline__ void stream_tiles(const StreamRows &A, v4i (&af)[KS], const int8_t *s_w,
                                             const int32_t *s_par, int8_t *s_stage,
                                             const Epilogue &ep, int M, int N, int n0,
                                             int bn, int tiles32, int first, int step, int lane) {
  constexpr int WSTRIDE = KS * 32 + 16, STRIDE = stream_stage_stride(NP);
  const int l32 = lane & 31, lhi = lane >> 5;
  int32_t lo, hi;
  activation_clamp(ep, lo, hi);
  const bool fast = fused_out_is_fast(ep);
  const FusedAddConsts fc = fused_add_consts(ep.add);
  const int8_t *w_lane = s_w + l32 * WSTRIDE + lhi * 16;
  // copy-out: lpr lanes per row, rpp rows per pass
  const int lpr = bn / 16, rpp = 64 / lpr;
  const int rb_row = lane / lpr, rb_seg = lane - rb_row * lpr;
  v4i an[KS];
  // (waited for here, once: inside the loop af is known to have arrived, and no
  // multiply waits behind the stores of the tile before)
#pragma unroll
  for (int ks = 0; ks < KS; ks++) asm volatile("" : "+v"(af[ks]));
  // The residual bytes of a tile, in the layout of the copy-out. A lane whose row
  // is past the tile or the end works on the tile's last row instead and stores the
  // same bytes to the same place as that row's own lane: with every load and store
  // issued by every lane the waits can be counted exactly.
  auto residual = [&](int t, int p) {
    const int m = t * 32 + min(p * rpp + rb_row, min(31, M - 1 - t * 32));
    return *reinterpret_cast<const int4 *>(ep.add.res + (long long)m * ep.ldc + n0 + rb_seg * 16);
  };
  int4 rq[NP];
  if constexpr (RES) {
#pragma unroll
    for (int p = 0; p < NP; p++) rq[p] = residual(min(first, tiles32 - 1), p);
  }
  for (int t = first; t < tiles32; t += step) {
    // (a wave's last tile once more behind it: the last tile of all would be asked for by
    // every wave at once)
    const int m0 = t * 32, next = t + step < tiles32 ? t + step : t;
    const int last_row = min(31, M - 1 - m0);      // of this tile
    // the next tile's rows are on their way while this one is worked on
    stream_load_rows<KS>(A, an, next, M, lane);
    for (int j = 0; j < bn / 32; j++) {
      const int cl = j * 32 + 16 * lhi;
      v16i acc = stream_acc_start<MODE>(s_par + cl);
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        const v4i b = *reinterpret_cast<const v4i *>(w_lane + j * 32 * WSTRIDE + ks * 32);
        // weights first: the result's rows are columns of the output
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(b, af[ks], acc, 0, 0, 0);
      }
      const int4 v = requant_pack16<MODE, LEAKY, kStreamBN, true>(acc, s_par + cl, ep, lo, hi);
      *reinterpret_cast<int4 *>(s_stage + l32 * STRIDE + cl) = v;
    }
    wave_fence();
#pragma unroll
    for (int p = 0; p < NP; p++) {
      const int row = min(p * rpp + rb_row, last_row), m = m0 + row;
      int4 v = *reinterpret_cast<const int4 *>(s_stage + row * STRIDE + rb_seg * 16);
      if constexpr (RES) {
        v = fused_out_words_loaded(v, rq[p], true, ep, fc, fast);
        rq[p] = residual(next, p);   // a whole tile ahead of its use
      } else {
        v = fused_out_words_loaded(v, v, false, ep, fc, fast);
      }
      *reinterpret_cast<int4 *>(ep.out + (long long)m * ep.ldc + n0 + rb_seg * 16) = v;
    }
    wave_fence();
#pragma unroll
    for (int ks = 0; ks < KS; ks++) af[ks] = an[ks];
  }
}

// K = 256: the plain form of the loop. A lane's rows alone are 32 registers
// there; with the next tile's rows and residual bytes asked for ahead
// the loop needs more registers than three waves per SIMD leave (spills, whose
// reloads wait behind the stores), and at two waves per SIMD it is slower than
// this: rows asked for at the top of the tile, the residual where it is added,
// four or five waves per SIMD as the LDS allows.
template <int KS, int NP, int MODE, bool LEAKY>
__device__ __forceinline__ void stream_tiles_simple(const StreamRows &A, const int8_t *s_w,
                                             const int32_t *s_par, int8_t *s_stage,
                                             const Epilogue &ep, int M, int N, int n0, int bn,
                                             int tiles32, int first, int step, int lane) {
  constexpr int WSTRIDE = KS * 32 + 16, STRIDE = stream_stage_stride(NP);
  const int l32 = lane & 31, lhi = lane >> 5;
  int32_t lo, hi;
  activation_clamp(ep, lo, hi);
  const bool fast = fused_out_is_fast(ep);
  const FusedAddConsts fc = fused_add_consts(ep.add);
  const int8_t *w_lane = s_w + l32 * WSTRIDE + lhi * 16;
  for (int t = first; t < tiles32; t += step) {
    const int m0 = t * 32;
    // rows past the end re-read the last row; their results are not stored
    const int8_t *ar = A.row(min(m0 + l32, M - 1)) + lhi * 16;
    v4i af[KS];
    if (A.seg_chunks >= KS) {
#pragma unroll
      for (int ks = 0; ks < KS; ks++) af[ks] = *reinterpret_cast<const v4i *>(ar + ks * 32);
    } else {
#pragma unroll
      for (int ks = 0; ks < KS; ks++) af[ks] = *reinterpret_cast<const v4i *>(ar + A.chunk(ks));
    }
    for (int j = 0; j < bn / 32; j++) {
      const int cl = j * 32 + 16 * lhi;
      v16i acc = stream_acc_start<MODE>(s_par + cl);
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        const v4i b = *reinterpret_cast<const v4i *>(w_lane + j * 32 * WSTRIDE + ks * 32);
        // weights first: the result's rows are columns of the output
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(b, af[ks], acc, 0, 0, 0);
      }
      const int4 v = requant_pack16<MODE, LEAKY, kStreamBN, true>(acc, s_par + cl, ep, lo, hi);
      *reinterpret_cast<int4 *>(s_stage + l32 * STRIDE + cl) = v;
    }
    wave_fence();
    wave_rows_copy_out(s_stage, STRIDE, bn, lane, m0, M, n0, ep, fc, fast);
    wave_fence();
  }
}

// Workgroups of four waves per CU, as many as the registers allow (66 to 132 of them; LDS may
// allow fewer). One kernel per number of copy-out passes, residual and requantisation
// variant: with all of them behind branches in one it was three for K of 64 and 128, four
// for 256. us, hinted, with the residual unless noted, before / now: 8 x 56x56 64 -> 256
// 9.2 / 8.8, 16 x 28x28 128 -> 512 10.6 / 10.0, 64 x 28x28 128 -> 512 25.5 / 24.2, without:
// 64 x 56x56 256 -> 128 22.4 / 21.6, 8 x 56x56 64 -> 64 4.4 / 4.0; 32 x 56x56 64 -> 256 with
// it 21.9 / 22.3, 64 x 28x28 128 -> 512 without 16.2 / 16.5 (1.2 and 1.5 tiles to a wave).
// At K = 64 with the residual two of the variants spill one and three registers for the fifth
// workgroup; with four, and no spill, they are level or behind (64 x 56x56 64 -> 256 33.4 with
// five, 34.0 with four, 64 -> 64 12.5 and 12.7, 64 -> 128 19.3 and 19.3).
template <int KS, bool RES, int MODE> constexpr int stream_per_cu() {
  constexpr bool full = RES && (KS == 3 || KS == 4);
  return MODE == 0 ? (full ? 3 : 4) : (full ? 4 : 5);
}

// KS: K / 32 (1 to 4, or 8). blockIdx.y: column slice of bn columns. MODE: requant_mode.
template <int KS, int NP, bool RES, int MODE, bool LEAKY>
__global__ __launch_bounds__(256, (stream_per_cu<KS, RES, MODE>())) void gemm_i8_stream_kernel(
    StreamRows A, const int8_t *W, Epilogue ep, int M, int N, int bn, int tiles32) {
  constexpr int K = KS * 32, WSTRIDE = K + 16, kStage = 32 * stream_stage_stride(NP);
  extern __shared__ __attribute__((aligned(16))) int8_t lds[];
  int32_t *s_par = reinterpret_cast<int32_t *>(lds);
  int8_t *s_stage = lds + kStreamParBytes;               // one tile per wave
  int8_t *s_w = s_stage + 4 * kStage;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = blockIdx.y * bn;
  const int cols = min(bn, N - n0);          // a multiple of 32

  // the wave's first rows are asked for before anything else, so that they
  // arrive while the slice is being put in LDS
  const int first = blockIdx.x * 4 + wave, step = gridDim.x * 4;
  v4i af[KS];
  if constexpr (KS < 8) stream_load_rows<KS>(A, af, min(first, tiles32 - 1), M, lane);

  // the slice's constants and weights -> LDS, once
  if (tid < cols) {
    ColRaw col[1];
    load_col_raw<1, kStreamBN>(col, ep, N, n0, 0, 0, tid);
    par_table_store<kStreamBN>(s_par, tid, col[0], ep, K, MODE);
  }
  {
    constexpr int CH = K / 16;               // 16-byte chunks per weight row
    const int chunks = cols * CH;
    const int8_t *w0 = W + (long long)n0 * K;
    for (int base = 0; base < chunks; base += 256 * 4) {
      int4 v[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int c = min(base + tid + u * 256, chunks - 1);
        v[u] = *reinterpret_cast<const int4 *>(w0 + (long long)c * 16);
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int c = base + tid + u * 256;
        if (c < chunks) {
          const int row = c / CH, kc = c - row * CH;
          *reinterpret_cast<int4 *>(s_w + perm_slot16(row) * WSTRIDE + kc * 16) = v[u];
        }
      }
    }
  }
  __syncthreads();

  // from here on every wave is on its own
  int8_t *stage = s_stage + wave * kStage;
  if constexpr (KS == 8)
    stream_tiles_simple<KS, NP, MODE, LEAKY>(A, s_w, s_par, stage, ep, M, N, n0, cols, tiles32, first,
                                         step, lane);
  else
    stream_tiles<KS, NP, RES, MODE, LEAKY>(A, af, s_w, s_par, stage, ep, M, N, n0, cols, tiles32,
                                           first, step, lane);
}

int gemm_stream_launch(const StreamRows &A, const int8_t *W, const Epilogue &ep, int M,
                       int N, int K, hipStream_t st) {
  // 128 columns per slice: a slice's weights stay under 35 KB beside 18 KB of
  // staging tiles and the 5 KB constants table, and a unit of work (32 rows of
  // one slice) is small enough that the last round of tiles, which only some of
  // the waves take part in, costs little (K = 64, 256 output columns, 200704
  // rows: 37.7 us in slices of 128 against 38.6 us in one of 256, though the
  // rows are then read twice)
  const int bn = 128;
  const int slices = (N + bn - 1) / bn;
  const size_t lds = (size_t)kStreamParBytes + 4 * 32 * (size_t)stream_stage_stride(N <= 64 ? 2 : 4) +
                     (size_t)std::min(bn, N) * (K + 16);
  const int tiles32 = (M + 31) / 32;
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
      cus = v;
  }
  MI355X_REQUIRE(slices < 65536, "problem too large");
  // variant by variant: K, passes of the copy-out (two for up to 64 columns), residual,
  // requantisation
  using std::integral_constant;
  auto launch = [&](auto ks, auto np, auto res, auto mode, auto leaky) {
    constexpr int most = stream_per_cu<ks.value, res.value, mode.value>();
    auto kernel = gemm_i8_stream_kernel<ks.value, np.value, res.value, mode.value, leaky.value>;
    const int per_cu = (int)std::min<size_t>(most, (160 * 1024) / lds);
    long long gx = std::max(1LL, (long long)cus * per_cu / slices);
    gx = std::min<long long>(gx, (tiles32 + 3) / 4);
    if (ks.value == 8) {
      // 128 columns x 272 bytes of weights: past the 48 KiB a launch gets unasked
      static std::atomic<uint64_t> attr_set{0};
      const int rc = set_lds_attr(kernel, 64 * 1024, attr_set);
      if (rc != MI355X_OK) return rc;
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)gx, (unsigned)slices), dim3(256), lds, st, A, W, ep, M,
                       N, bn, tiles32);
    return check_launch("gemm_i8_stream");
  };
  auto with_mode = [&](auto ks, auto np, auto res) {
    using No = std::false_type;
    if (ep.act == 5) return launch(ks, np, res, integral_constant<int, 0>{}, std::true_type{});
    if ((ep.fast & 3) == 3) return launch(ks, np, res, integral_constant<int, 3>{}, No{});
    if (ep.fast & 1) return launch(ks, np, res, integral_constant<int, 1>{}, No{});
    return launch(ks, np, res, integral_constant<int, 0>{}, No{});
  };
  auto with_passes = [&](auto ks) {
    using Two = integral_constant<int, 2>;
    using Four = integral_constant<int, 4>;
    const bool narrow = N <= 64;
    if (ep.add.res)
      return narrow ? with_mode(ks, Two{}, std::true_type{}) : with_mode(ks, Four{}, std::true_type{});
    return narrow ? with_mode(ks, Two{}, std::false_type{}) : with_mode(ks, Four{}, std::false_type{});
  };
  switch (K) {
  case 32: return with_passes(integral_constant<int, 1>{});
  case 64: return with_passes(integral_constant<int, 2>{});
  case 96: return with_passes(integral_constant<int, 3>{});
  case 128: return with_passes(integral_constant<int, 4>{});
  default:     // (the plain loop asks for the residual where it adds it)
    return N <= 64 ? with_mode(integral_constant<int, 8>{}, integral_constant<int, 2>{}, std::false_type{})
                   : with_mode(integral_constant<int, 8>{}, integral_constant<int, 4>{}, std::false_type{});
  }
}

} // namespace mi355x
