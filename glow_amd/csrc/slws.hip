// FusedRowwiseQuantizedSparseLengthsWeightedSum / Sum and the offsets-based
// EmbeddingBag twin, for 8-bit and 4-bit fused rows with fp32 or fp16
// scale/offset (reference lib/LLVMIRCodeGen/libjit/libjit.cpp:1253-1276,
// 2454-2481; lib/Backends/Interpreter/InterpreterNodes.cpp:5764-5889).
//
// One bag per group of LPB lanes (a whole 64-lane wavefront for rows of 64+
// data bytes, so every row read is one coalesced request). A lane owns BPL
// consecutive data bytes of the row and keeps their running sums in
// registers. For each batch of up to 64 lookups lane j first fetches index j,
// weight j and the (scale, offset) pair of row j; then all row reads of the
// batch are issued back to back before the first one is consumed, so a bag
// costs three dependent memory round trips however long it is. The sums are
// formed in bag order with separately rounded multiply and add, which
// reproduces the CPU loop bit for bit.
//
// In the wavefront-per-bag kernel the per-lookup values (row byte offset,
// weight, scale, offset) are handed from lane j to the whole wave through a
// wave-private LDS slot read back at a uniform address (a broadcast), which
// keeps the vector ALU for the five operations per element the arithmetic
// needs (convert, multiply, add, multiply, add).
//
// That is the strict form of the arithmetic (slws_kernel, slws_wave_kernel;
// MI355X_SLWS_MATH_STRICT). By default rows of 32 to 256 data bytes (a multiple
// of 4, in rows that start on a word) with fp32 accumulation run the fused
// kernels further down (slws_rows_kernel,
// slws_groups_kernel): the CPU loop's own expression per element, with two fused
// multiply-adds (MI355X_SLWS_MATH_ELEMENT), summed in bag order or in two, four or
// eight parts that are (as many rows as a wavefront's load fetches), or on request the
// sum regrouped into one fused multiply-add per element (_REGROUPED). A call
// names its arithmetic in mi355x_launch_opts; mi355x_slws_set_fused_math sets
// what the calls that name none get.
//
// The start of a bag in the index list is the exclusive prefix sum of the
// lengths. A block sums the lengths in front of it itself (from the start of
// its chunk of bags, plus one pre-summed value per earlier chunk),
// which keeps the common small-batch case at a single launch.
#include "common.h"

// Every multiply and add below must round on its own (the CPU code this
// reproduces has no fused multiply-add). The pragma covers contraction in the
// front end; the build must also pass -ffp-contract=off (the Makefile does),
// because HIP's default "fast" mode fuses in the back end regardless.
#pragma clang fp contract(off)

#include <hip/hip_fp16.h>

#include <atomic>
#include <type_traits>
#include <mutex>
#include <vector>

namespace mi355x {

constexpr int kSlwsThreads = 256;
constexpr int kBatch = 64;         // lookups fetched per round
// Up to kOneChunkBags bags a block sums the lengths in front of it itself, all of
// them in one memory trip. Beyond, a pre-pass sums chunks of kChunkBags bags and a
// block only its own chunk's: fewer bytes per block for a launch more, which with
// the wait for it costs 5 us (8192 bags of 40 rows of 128 bytes 17.5 -> 11.2 us,
// 16 000 bags 26.5 -> 20.3 us without it; at 17 000 the two are level).
constexpr int kOneChunkBags = 16384;
constexpr int kChunkBags = 4096;
constexpr int kTableBags = 4096;   // bags per table of a multi-table launch
constexpr int kMaxChunks = 32768;  // workspace entries (int64 each)
// Bags per block of slws_rows_kernel. At 4096 bags sixteen (one block of 1024
// threads per CU: the lengths in front of a block are summed once per CU), eight
// from kRowsWideBags on (measured: 3 % faster at 4096 bags, level at 16 384, 6 %
// slower at 65 536; reached by the launches that slws_ranges_kernel does not take: long bags
// (kRangesLen4, kRangesLen128), several tables, tables past 4 GB, the regrouped arithmetic), and
// below kRowsFewBags four, so that a small launch is spread over the CUs instead of filling a few
// of them.
constexpr int kRowsWaves = 16, kRowsWavesMany = 8, kRowsWavesFew = 4;
constexpr size_t kRowsWideBags = 16384, kRowsFewBags = 2048;
__host__ __device__ constexpr int rows_waves(size_t bags) {
  return bags < kRowsFewBags ? kRowsWavesFew : bags < kRowsWideBags ? kRowsWaves : kRowsWavesMany;
}
// Rows of up to 64 data bytes run with a bag per wavefront up to this many bags
// per launch (its lookups side by side in the lanes: the launch is as long as one
// bag's chain of dependent operations), several bags per wavefront beyond, where
// the instructions a wavefront issues bound it. 64 columns of four bits, 20 lookups
// a bag: 1000 bags 7.7 -> 3.8 us, 8000 bags 15.0 -> 6.8 (9.6 of it the second launch
// and the form with several bags); several bags from here on: 16 000 bags 11.4.
constexpr size_t kShortRowsWaveBags = 12288;
static_assert(kShortRowsWaveBags <= kRowsWideBags, "short rows have no eight-wave form");
// Rows of less than 32 data bytes take a lane per byte up to this many bags (16
// columns, 1000 bags: 9.7 us before, 10.1 with a lane per four bytes, 4.9), a lane
// per four bytes beyond.
constexpr size_t kByteLaneBags = 16384;
// slws_wide_kernel: from more than this many bags on, of rows of 65 to 128 bytes that start
// on a word at most this many lookups and data bytes on the average, and its lines for rows
// at any byte. A bag longer than kLongBag and than kLongBagMeans times the average gets a
// wavefront of its own there: side by side with its neighbours it goes on at 100 ns a lookup,
// alone at 27 (128 columns, 13 000 bags of 4, one of 1000 31 / 91 us, one of 5000 142 / 501,
// the kernels that take a bag per wavefront / this one before it did so; 30 and 140 now).
constexpr size_t kWideBags = 12288, kWideLen = 9, kWideBytes = 900, kWideAnyBags = 24000,
                 kWideAnyLen = 16, kLongBag = 32, kLongBagMeans = 4;

// slws_ranges_kernel takes rows of more than 64 bytes from so many bags on that the kernel for
// a bag per wavefront, which holds 4096 (8192 with up to 64 registers) at once, is behind: its
// last few blocks still find room (us, rows / ranges: 128 columns fp16 scales 4097 x 20 5.5 / 5.7,
// 4112 6.7 / 5.6; 256 columns 4097 x 6 5.2 / 5.5, 4112 6.0 / 5.5), longest of rows of four bits
// (200 columns 4097 x 6 5.2 / 7.1, 4160 x 20 9.9 / 9.1, 400 columns 4128 x 6 7.6 / 8.0) and of up to
// 128 bytes with fp32 scales (100 columns 4128 x 6 4.7 / 5.2, 4160 x 20 6.3 / 6.5, 4400 x 45 10.2 / 10.0).
// Rows of more than 128 bytes and bags of kRangesLenWide of them fill the chip earlier (256 columns 4097 x
// 15 7.1 / 6.6, x 30 9.6 / 8.5; four bits 400 columns 4112 x 20 13.3 / 12.6, 4097 10.3 / 12.5).
// Of rows of up to 128 bytes (eight bits with fp16 scales apart, which take a register more) not between
// kRangesBags64 and kRangesBags128: there two blocks of slws_rows_kernel to a CU hold every bag at once, and
// sixteen bags to eight wavefronts go in two turns (us, rows / ranges, 128 columns 6500 x 20
// 6.3 / 6.8, 8192 x 8 5.5 / 6.2; but 5000 x 60 12.4 / 10.5, 8300 x 80 20.6 / 18.1; 100 columns 8193 x 30
// 9.2 / 10.0, 8256 11.2 / 11.0; four bits 200 columns 8193 x 30 13.8 / 14.8, 8224 16.5 / 14.6). 768
// blocks of eight wavefronts are resident with eight-bit rows (67 to 73 registers) and four-bit ones of up
// to 128 bytes with fp16 scales (75), 512 with the other four-bit ones (81). A block's share is rounded up
// to whole turns of its wavefronts, of four-bit rows, of which a turn is longer, only to four bags (200
// columns x 30, whole turns / four: 8704 bags 16.2 / 14.7, 9500 16.2 / 14.9, 13 500 20.1 / 18.3; eight bits
// 200 columns x 30 7000 bags 13.0 / 14.3, 12 289 17.5 / 19.4, 13 500 21.1 / 19.6); 768 blocks in place of
// 512 of four bits and 200 columns 6000 x 30 11.9 / 10.3, 30 000 x 10 22.4 / 20.9.
// Long bags: four bits 200 columns, 17 623 x 80 46.6 / 49.8, x 145 71 / 78, 9000 x 145 48.4 /
// 50.0, but x 40 20.8 / 19.1; eight bits 100 columns 17 623 x 145 48.1 / 51.3, but x 80 33.2 /
// 32.4, 5000 x 145 23.8 / 19.5; wider ones of eight bits stay ahead, 200 columns 17 623 x 145
// 76.5 / 71.9.
constexpr size_t kRangesLen4 = 64, kRangesLen128 = 112;
constexpr int kRangesWaves = 8;
constexpr size_t kRangesBagsEarly = 4096, kRangesBags = 4111, kRangesBagsLate = 4159, kRangesLenWide = 12,
                 kRangesBags64 = 6144, kRangesBags128 = 8223, kRangesBlocks = 768, kRangesBlocks4 = 512;
// Bags up to which its blocks sum all lengths in front of them, without the launch that sums
// chunks: they are few, so that the lengths come from L2 some 400 times, not a few thousand. us,
// with that launch / without, x 30: 100 columns 17 000 18.3 / 16.2, 30 000 24.4 / 22.5, 40 000
// 30.6 / 29.3, 48 000 34.3 / 33.6; 256 columns 30 000 37.0 / 35.2, 48 000 64.4 / 63.5; four bits
// 200 columns 20 000 25.0 / 23.3, 40 000 41.4 / 40.8; 128 columns x 12 20 000 14.6 / 13.1,
// 48 000 22.7 / 23.1; past 49 152 each compute unit has twice the blocks (65 000 x 30 48.0 / 52.7).
constexpr int kRangesOneBags = 40960;
static_assert(kRangesOneBags % 4 == 0 && kRangesOneBags >= kOneChunkBags, "wave_before_long");

struct SlwsArgs {
  void *dest;
  const uint8_t *data;
  const void *weights;     // fp32 / fp16 / NULL
  const void *indices;     // int64 / int32
  const int32_t *lengths;  // lengths mode
  const int32_t *offsets;  // offsets mode (NULL in lengths mode)
  const int64_t *chunk_sums; // lengths mode with more than one chunk
  int64_t data_rows;
  int64_t num_indices;
  int64_t segments;        // number of output rows
  int32_t offsets_have_end;
  int32_t in_line;         // bytes per fused row
  int32_t data_bytes;      // quantized bytes per row (before scale/offset)
  int32_t out_cols;
  int32_t out16, w16, idx64;
  // rowwise (not fused) tables: scale and offset of row r are sep_scales[r],
  // sep_offsets[r] (fp32) and rows hold data bytes only
  const float *sep_scales, *sep_offsets;
  // multi-table launches: blockIdx.y selects the table whose pointers replace
  // the ones above
  const mi355x_sls_table *tables;
  // output transform: 0 = fp32 / fp16 rows as above; 1 = round to fp16 when
  // out16 (what the operator stores), then Quantize to int8 with (q_scale,
  // q_offset), rows q_stride bytes apart (ConvertTo + Quantize + InsertTensor
  // behind the lookup)
  int32_t out_q8;
  float q_scale, q_offset;
  int64_t q_stride;
  int32_t long_bag;        // slws_wide_kernel: longer bags take a wavefront of their own
};

__device__ __forceinline__ void select_table(SlwsArgs &a) {
  if (a.tables) {
    const mi355x_sls_table t = a.tables[blockIdx.y];
    a.data = t.data;
    a.indices = t.indices;
    a.lengths = t.lengths;
    a.offsets = t.bag_offsets;
    a.offsets_have_end = 1;
    a.dest = t.dest;
    a.data_rows = (int64_t)t.data_rows;
    a.num_indices = (int64_t)t.num_indices;
  }
}

// Stores the columns [col0, col0 + N) of output row `bag`; a lane's 4 or 8
// columns leave as one store when all of them exist and the address allows
// (as N byte or half-word stores they were N memory instructions per lane).
template <int N>
__device__ __forceinline__ void store_columns(const SlwsArgs &a, long long bag, int col0,
                                              const float (&acc)[N]) {
  if (a.out_q8) {
    int8_t *d = reinterpret_cast<int8_t *>(a.dest) + bag * a.q_stride + col0;
    uint32_t packed[(N + 3) / 4] = {};
#pragma unroll
    for (int c = 0; c < N; c++) {
      const float v = a.out16 ? __half2float(__float2half_rn(acc[c])) : acc[c];
      // the Quantize kernel's expression (the conversion saturates)
      const float r = rintf(__fadd_rn(__fdiv_rn(v, a.q_scale), a.q_offset));
      packed[c / 4] |= (uint32_t)(min(max((int32_t)r, -128), 127) & 0xff) << (8 * (c & 3));
    }
    if (N % 4 == 0 && col0 + N <= a.out_cols && ((((uintptr_t)d) & (N - 1)) == 0)) {
      if constexpr (N == 8) *reinterpret_cast<uint2 *>(d) = make_uint2(packed[0], packed[1]);
      if constexpr (N == 4) *reinterpret_cast<uint32_t *>(d) = packed[0];
    } else {
#pragma unroll
      for (int c = 0; c < N; c++)
        if (col0 + c < a.out_cols) d[c] = (int8_t)(packed[c / 4] >> (8 * (c & 3)));
    }
    return;
  }
  const long long o0 = bag * (long long)a.out_cols + col0;
  if (a.out16) {
    __half *d = reinterpret_cast<__half *>(a.dest) + o0;
    uint32_t packed[(N + 1) / 2] = {};
#pragma unroll
    for (int c = 0; c < N; c++)
      packed[c / 2] |= (uint32_t)__half_as_ushort(__float2half_rn(acc[c])) << (16 * (c & 1));
    if (N % 4 == 0 && col0 + N <= a.out_cols && ((((uintptr_t)d) & (2 * N - 1)) == 0)) {
      if constexpr (N == 8)
        *reinterpret_cast<uint4 *>(d) = make_uint4(packed[0], packed[1], packed[2], packed[3]);
      if constexpr (N == 4) *reinterpret_cast<uint2 *>(d) = make_uint2(packed[0], packed[1]);
    } else {
#pragma unroll
      for (int c = 0; c < N; c++)
        if (col0 + c < a.out_cols)
          d[c] = __ushort_as_half((unsigned short)(packed[c / 2] >> (16 * (c & 1))));
    }
  } else {
    float *d = reinterpret_cast<float *>(a.dest) + o0;
    if constexpr (N % 4 == 0) {
      if (col0 + N <= a.out_cols && ((((uintptr_t)d) & 15) == 0)) {
#pragma unroll
        for (int c = 0; c < N; c += 4)
          *reinterpret_cast<float4 *>(d + c) =
              make_float4(acc[c], acc[c + 1], acc[c + 2], acc[c + 3]);
        return;
      }
    }
    if (N == 2 && col0 + 1 < a.out_cols && ((((uintptr_t)d) & 7) == 0)) {
      *reinterpret_cast<float2 *>(d) = make_float2(acc[0], acc[N - 1]);
    } else {
#pragma unroll
      for (int c = 0; c < N; c++)
        if (col0 + c < a.out_cols) d[c] = acc[c];
    }
  }
}

typedef uint8_t __attribute__((address_space(1))) global_u8;
typedef unsigned short __attribute__((address_space(1))) global_u16;

template <int LPB> __device__ __forceinline__ int bcast_i(int v, int j) {
  if constexpr (LPB == 64) {
    return __builtin_amdgcn_readlane(v, j);
  } else {
    return __shfl(v, j, LPB);
  }
}
template <int LPB> __device__ __forceinline__ float bcast_f(float v, int j) {
  return __int_as_float(bcast_i<LPB>(__float_as_int(v), j));
}

__device__ __forceinline__ uint32_t load_u32_any(const uint8_t *p) {
  if ((((uintptr_t)p) & 3) == 0) return *reinterpret_cast<const uint32_t *>(p);
  return (uint32_t)p[0] | ((uint32_t)p[1] << 8) | ((uint32_t)p[2] << 16) |
         ((uint32_t)p[3] << 24);
}

__device__ __forceinline__ float f16round(float v) {
  return __half2float(__float2half_rn(v));
}

// acc += w * (scale * q + offset), each operation rounded on its own; with
// fp16 accumulation the product and the sum are rounded to binary16 the way
// glow::float16's operator+= does (reference include/glow/Support/Float16.h).
template <bool ACC16>
__device__ __forceinline__ float accumulate(float acc, float w, float s,
                                            float o, uint32_t q) {
  float d = __fadd_rn(__fmul_rn(s, (float)q), o);
  float t = __fmul_rn(d, w);
  if constexpr (ACC16) {
    // The product must be rounded to binary32 before it is rounded to
    // binary16, as on the CPU. Left to itself the compiler merges multiply and
    // conversion into one mixed-precision operation that rounds once, which
    // differs in the last place now and then; the empty statement keeps the
    // binary32 product as a value of its own.
    asm volatile("" : "+v"(t));
    return f16round(__fadd_rn(acc, f16round(t)));
  } else {
    return __fadd_rn(acc, t);
  }
}

// Sum of v over the 64 lanes of the wave, returned wave-uniform. Lanes are
// combined inside each row of 16 with DPP moves (no LDS round trip), the four
// row totals are read out as scalars.
__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t v) {
  int x = (int)v;
  x += __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xf, 0xf, true);  // quad_perm [1,0,3,2]
  x += __builtin_amdgcn_update_dpp(0, x, 0x4E, 0xf, 0xf, true);  // quad_perm [2,3,0,1]
  x += __builtin_amdgcn_update_dpp(0, x, 0x141, 0xf, 0xf, true); // row_half_mirror
  x += __builtin_amdgcn_update_dpp(0, x, 0x140, 0xf, 0xf, true); // row_mirror
  return (uint32_t)__builtin_amdgcn_readlane(x, 0) +
         (uint32_t)__builtin_amdgcn_readlane(x, 16) +
         (uint32_t)__builtin_amdgcn_readlane(x, 32) +
         (uint32_t)__builtin_amdgcn_readlane(x, 48);
}

// Inclusive prefix sum of v over the 64 lanes of the wave: shifts inside rows of
// 16 lanes, then the totals of the rows in front (DPP moves only).
__device__ __forceinline__ uint32_t wave_scan_u32(uint32_t v) {
  int x = (int)v;
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false); // row_bcast:15 into rows 1, 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false); // row_bcast:31 into rows 2, 3
  return (uint32_t)x;
}

__device__ __forceinline__ uint32_t clamp_len(int v) {
  return v > 0 ? (uint32_t)v : 0u;
}
// v into [0, most] (most not negative and the same in every lane), one instruction
__device__ __forceinline__ uint32_t clamp_len(int v, int most) {
  uint32_t r;
  asm("v_med3_i32 %0, %1, 0, %2" : "=v"(r) : "v"(v), "s"(most));
  return r;
}

// A bag starts where the lengths in front of it say, or is empty where that is at or
// past the end of the index list. So no sum needs to go past num_indices: with lists
// of less than 2^26 lookups every length, every thread's sum, every wave's sum is
// cut off there, and 32 bits hold what the next step adds up (64 of them, or sixteen
// partial sums and sixteen lengths), whatever the lengths are. Longer lists are
// summed in 64 bits.
constexpr int kNarrowBits = 26;
__device__ __forceinline__ bool narrow_list(const SlwsArgs &a) {
  return __builtin_expect(((uint64_t)a.num_indices >> kNarrowBits) == 0, 1);   // scalar
}

// Offsets mode: span of `bag` read off the offsets vector.
__device__ __forceinline__ void bag_span_offsets(const SlwsArgs &a,
                                                 long long bag,
                                                 long long &start, int &len) {
  start = 0;
  len = 0;
  if (bag < a.segments) {
    // both ends are clamped into the index list, so that offsets that make no
    // sense (negative, decreasing, past the end) give short or empty bags and
    // never a position outside the list
    start = min(max((long long)a.offsets[bag], 0LL), (long long)a.num_indices);
    long long end = (!a.offsets_have_end && bag == a.segments - 1)
                        ? a.num_indices
                        : (long long)a.offsets[bag + 1];
    end = min(max(end, start), (long long)a.num_indices);
    len = (int)min(end - start, 0x7fffffffLL);
  }
}

// (four lengths in one request wherever they start: one table's slice of a [tables x batch]
// tensor of an odd batch starts on any of them)
typedef int __attribute__((ext_vector_type(4))) i32x4;
typedef i32x4 __attribute__((aligned(4))) i32x4_any;
typedef i32x4_any __attribute__((address_space(1))) global_i32x4;

// One thread's share of the sum of the clamped lengths p[0 .. 4 * nvec): TRIPS
// requests of four, all in flight together (positions past the end re-read the
// last four and are masked out: a request under a condition of its own is waited
// for on its own).
template <int TRIPS, int THREADS>
__device__ __forceinline__ uint32_t sum_lengths_trips(const global_i32x4 *l4, int nvec, int tid,
                                                      int most) {
  i32x4 x[TRIPS];
#pragma unroll
  for (int u = 0; u < TRIPS; u++) x[u] = l4[min(tid + u * THREADS, nvec - 1)];
  if constexpr (TRIPS > 1) __builtin_amdgcn_sched_barrier(0);
  uint32_t part = 0;
#pragma unroll
  for (int u = 0; u < TRIPS; u++) {
    const uint32_t t = clamp_len(x[u].x, most) + clamp_len(x[u].y, most) + clamp_len(x[u].z, most) +
                       clamp_len(x[u].w, most);
    part += (tid + u * THREADS < nvec) ? t : 0u;
  }
  return part;
}

// The same for up to kOneChunkBags lengths, by how many trips they need (nvec is
// uniform).
template <int THREADS>
__device__ __forceinline__ uint32_t sum_lengths(const int32_t *p, int nvec, int tid, int most) {
  const global_i32x4 *l4 = (const global_i32x4 *)p;
  constexpr int kMost = kOneChunkBags / 4 / THREADS;
  if (nvec == 0) return 0;
  if (nvec <= THREADS) return sum_lengths_trips<1, THREADS>(l4, nvec, tid, most);
  if constexpr (kMost > 4)
    if (nvec <= 4 * THREADS) return sum_lengths_trips<4, THREADS>(l4, nvec, tid, most);
  return sum_lengths_trips<kMost, THREADS>(l4, nvec, tid, most);
}

// What this wave's threads see of the clamped lengths in front of the block (n of them
// from p on: less than kOneChunkBags, a multiple of 4) and of the sums of the chunks
// before p's: their sum, cut off at `most` = num_indices < 2^26.
template <int THREADS>
__device__ __forceinline__ uint32_t wave_before(const int32_t *p, int n, const int64_t *chunk_sums,
                                                int chunk, int tid, int most) {
  static_assert(kOneChunkBags / THREADS <= 64, "a thread's lengths add up in 32 bits");
  uint32_t part = min(sum_lengths<THREADS>(p, n >> 2, tid, most), (uint32_t)most);
  if (chunk_sums)
    for (int c = tid; c < chunk; c += THREADS)
      part = min(part + (uint32_t)min((long long)chunk_sums[c], (long long)most), (uint32_t)most);
  return min(wave_sum_u32(part), (uint32_t)most);
}
// The same for any number of lengths and no chunks, kOneChunkBags of them to a trip (sixteen loads a
// thread and trip in place of eight take 111 registers). us, lengths that start off sixteen bytes
// one by one / four to a request, as on sixteen: 100 columns x 20 5000 bags 8.1 / 7.1, 16 000 17.3 / 13.0,
// 40 000 37.3 / 25.4; 256 columns x 12 40 000 40.6 / 28.0.
template <int THREADS>
__device__ __forceinline__ uint32_t wave_before_long(const int32_t *p, int n, int tid, int most) {
  uint32_t part = 0;
  for (int at = 0; at < n; at += kOneChunkBags)
    part = min(part + min(sum_lengths<THREADS>(p + at, min(n - at, kOneChunkBags) >> 2, tid, most),
                          (uint32_t)most),
               (uint32_t)most);
  return min(wave_sum_u32(part), (uint32_t)most);
}
// The same in 64 bits (n a multiple of 4).
template <int THREADS>
__device__ __forceinline__ long long wave_before_wide(const int32_t *p, int n, const int64_t *chunk_sums,
                                                      int chunk, int tid) {
  const global_i32x4 *l4 = (const global_i32x4 *)p;
  long long sum = 0;
  for (int i = tid; i < n >> 2; i += THREADS) {
    const i32x4 x = l4[i];
    sum += (long long)clamp_len(x.x) + clamp_len(x.y) + clamp_len(x.z) + clamp_len(x.w);
  }
  if (chunk_sums)
    for (int c = tid; c < chunk; c += THREADS) sum += chunk_sums[c];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
  return sum;
}

// Lengths mode, first half: every wave leaves the sum of the clamped lengths
// it has seen in front of the block in s_part[wave], and the block's own
// clamped lengths go to s_own[]. Ends with a block barrier.
template <int kGroups, int kThreads = kSlwsThreads>
__device__ __forceinline__ void block_prefix(const SlwsArgs &a, int tid,
                                             long long first_bag,
                                             long long *s_part, int *s_own) {
  const long long chunk = a.chunk_sums ? first_bag / kChunkBags : 0;
  const long long lo = chunk * kChunkBags;
  const int32_t *lbase = a.lengths + lo;
  const int n_before = (int)(first_bag - lo); // < kOneChunkBags, multiple of 4
  const long long before =
      narrow_list(a)
          ? (long long)wave_before<kThreads>(lbase, n_before, a.chunk_sums, (int)chunk, tid,
                                             (int)a.num_indices)
          : wave_before_wide<kThreads>(lbase, n_before, a.chunk_sums, (int)chunk, tid);
  if (tid < kGroups) {
    const long long b = first_bag + tid;
    s_own[tid] = (int)min(clamp_len(b < a.segments ? a.lengths[b] : 0),
                          0x7fffffffu);
  }
  if ((tid & 63) == 0) s_part[tid >> 6] = before;
  __syncthreads();
}

// Position of the first lookup of `bag` in the index list and its length.
// Lengths mode: exclusive prefix sum of the clamped lengths in front of the
// block (summed by the block itself, all loads in one memory round trip) plus
// the lengths of the block's earlier bags; checked against num_indices before any
// use. Offsets mode: read off the offsets vector.
template <int kGroups>
__device__ __forceinline__ void bag_span(const SlwsArgs &a, int tid, int grp,
                                         long long bag, long long first_bag,
                                         long long *s_part, int *s_own,
                                         long long &start, int &len) {
  if (a.offsets) {
    bag_span_offsets(a, bag, start, len);
    return;
  }
  block_prefix<kGroups>(a, tid, first_bag, s_part, s_own);
  start = 0;
#pragma unroll
  for (int w = 0; w < kSlwsThreads / 64; w++) start += s_part[w];
  static_assert(kGroups <= 64, "one lane per bag of the block");
  const int lane = tid & 63;
  const int own = lane < kGroups ? s_own[lane] : 0;
  if (__ballot(own >= (1 << 25)) == 0) {
    // the lengths of the block's earlier bags as one scan over the lanes
    // (64 lengths below 2^25 stay inside 32 bits); read one by one they were up
    // to 31 dependent LDS loads
    const int before = (int)wave_scan_u32((uint32_t)own) - own;
    start += __shfl(before, grp, 64);
  } else {
    for (int g = 0; g < grp; g++) start += s_own[g];
  }
  len = bag < a.segments ? s_own[grp] : 0;
}

template <int LPB, int BPL, bool IS4, bool SO16, bool ACC16>
__global__ __launch_bounds__(kSlwsThreads) void slws_kernel(SlwsArgs a) {
  select_table(a);
  constexpr int kGroups = kSlwsThreads / LPB;      // bags per block
  constexpr int kColsPerByte = IS4 ? 2 : 1;
  constexpr int kColsPerLane = BPL * kColsPerByte;
  __shared__ long long s_part[kSlwsThreads / 64];
  __shared__ int s_own[kGroups];

  const int tid = threadIdx.x;
  const int sub = tid % LPB;                        // lane within the bag group
  const int grp = tid / LPB;
  const long long first_bag = (long long)blockIdx.x * kGroups;
  const long long bag = first_bag + grp;

  long long start = 0;
  int len = 0;
  bag_span<kGroups>(a, tid, grp, bag, first_bag, s_part, s_own, start, len);
  // a bag cannot use more lookups than the index list holds: bounds the loop
  // below whatever the lengths say
  {
    const long long room = a.num_indices - start;
    len = room <= 0 ? 0 : (int)min((long long)len, room);
  }

  const int n_passes = (a.data_bytes + LPB * BPL - 1) / (LPB * BPL);
  for (int pass = 0; pass < n_passes; pass++) {
    const int byte0 = (pass * LPB + sub) * BPL;       // first data byte of lane
    const bool lane_live = byte0 < a.data_bytes;
    float acc[kColsPerLane];
#pragma unroll
    for (int c = 0; c < kColsPerLane; c++) acc[c] = 0.0f;

    for (int base = 0; base < len; base += kBatch) {
      const int cnt = min(kBatch, len - base);
      // first pass: lookup `sub + k*LPB` of the batch is fetched by lane `sub`
      constexpr int kPerLane = kBatch / LPB;
      int row_lo[kPerLane];
      float wgt[kPerLane], scl[kPerLane], ofs[kPerLane];
#pragma unroll
      for (int k = 0; k < kPerLane; k++) {
        const int j = sub + k * LPB;
        long long pos = start + base + j;
        long long row = -1;
        float w = 0.0f;
        if (j < cnt && pos < a.num_indices) {
          row = a.idx64 ? reinterpret_cast<const long long *>(a.indices)[pos]
                        : (long long)reinterpret_cast<const int *>(a.indices)[pos];
          if (!a.weights) {
            w = 1.0f;
          } else if (a.w16) {
            w = __half2float(reinterpret_cast<const __half *>(a.weights)[pos]);
          } else {
            w = reinterpret_cast<const float *>(a.weights)[pos];
          }
        }
        float s = 0.0f, o = 0.0f;
        if (row >= 0 && row < a.data_rows) {
          const uint8_t *so = a.data + row * a.in_line + a.data_bytes;
          if constexpr (SO16) {
            uint32_t v = load_u32_any(so);
            s = __half2float(__ushort_as_half((unsigned short)(v & 0xffff)));
            o = __half2float(__ushort_as_half((unsigned short)(v >> 16)));
          } else if (a.sep_scales) {
            s = a.sep_scales[row];
            o = a.sep_offsets[row];
          } else {
            s = __uint_as_float(load_u32_any(so));
            o = __uint_as_float(load_u32_any(so + 4));
          }
        } else {
          row = 0; // skipped lookup: reads row 0, contributes w * 0
          w = 0.0f;
        }
        row_lo[k] = (int)row; // data_rows * in_line is checked to fit 2^31 rows
        wgt[k] = w;
        scl[k] = s;
        ofs[k] = o;
      }
      // second pass: all row reads of the batch in flight before the first use
      uint32_t q[kBatch];
#pragma unroll
      for (int j = 0; j < kBatch; j++) {
        q[j] = 0;
        if (j < cnt) {
          const int row = bcast_i<LPB>(row_lo[j / LPB], j % LPB);
          if (lane_live) {
            const uint8_t *p = a.data + (long long)row * a.in_line + byte0;
            if constexpr (BPL == 2) {
              q[j] = *reinterpret_cast<const unsigned short *>(p);
            } else {
              q[j] = *p;
            }
          }
        }
      }
#pragma unroll
      for (int j = 0; j < kBatch; j++) {
        if (j < cnt) {
          const float w = bcast_f<LPB>(wgt[j / LPB], j % LPB);
          const float s = bcast_f<LPB>(scl[j / LPB], j % LPB);
          const float o = bcast_f<LPB>(ofs[j / LPB], j % LPB);
#pragma unroll
          for (int b = 0; b < BPL; b++) {
            const uint32_t byte = (q[j] >> (8 * b)) & 0xff;
            if constexpr (IS4) {
              acc[2 * b] = accumulate<ACC16>(acc[2 * b], w, s, o, byte & 15);
              acc[2 * b + 1] = accumulate<ACC16>(acc[2 * b + 1], w, s, o, byte >> 4);
            } else {
              acc[b] = accumulate<ACC16>(acc[b], w, s, o, byte);
            }
          }
        }
      }
    }

    if (bag < a.segments && lane_live)
      store_columns<kColsPerLane>(a, bag, byte0 * kColsPerByte, acc);
  }
}

// Orders this wave's LDS writes before its later LDS reads of other lanes'
// slots. LDS operations of one wave execute in order; the fences keep the
// compiler from moving them across.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Span of the bag of one wavefront (4 waves, 4 consecutive bags per block),
// returned wave-uniform so that it stays in scalar registers. Lengths mode
// ends with a block barrier. A bag cannot use more lookups than the index list
// holds, which bounds the callers' loops whatever the lengths say.
__device__ __forceinline__ void wave_bag_span(const SlwsArgs &a, int tid, int wave,
                                              long long bag, long long first_bag,
                                              long long *s_part, int *s_own,
                                              long long &start, int &len) {
  constexpr int kGroups = 4;
  if (a.offsets) {
    long long start_v;
    int len_v;
    bag_span_offsets(a, bag, start_v, len_v);
    len = __builtin_amdgcn_readfirstlane(len_v);
    start = ((long long)__builtin_amdgcn_readfirstlane((int)(start_v >> 32)) << 32) |
            (unsigned int)__builtin_amdgcn_readfirstlane((int)start_v);
  } else {
    block_prefix<kGroups>(a, tid, first_bag, s_part, s_own);
    const long long block_start = s_part[0] + s_part[1] + s_part[2] + s_part[3];
    const int4 own = *reinterpret_cast<const int4 *>(s_own);
    const int w = __builtin_amdgcn_readfirstlane(wave);
    const int o0 = __builtin_amdgcn_readfirstlane(own.x);
    const int o1 = __builtin_amdgcn_readfirstlane(own.y);
    const int o2 = __builtin_amdgcn_readfirstlane(own.z);
    const int o3 = __builtin_amdgcn_readfirstlane(own.w);
    const long long bs =
        ((long long)__builtin_amdgcn_readfirstlane((int)(block_start >> 32)) << 32) |
        (unsigned int)__builtin_amdgcn_readfirstlane((int)block_start);
    start = bs + (w > 0 ? o0 : 0) + (w > 1 ? o1 : 0) + (w > 2 ? o2 : 0);
    len = w == 0 ? o0 : (w == 1 ? o1 : (w == 2 ? o2 : o3));
    if (bag >= a.segments) len = 0;
  }
  const long long room = a.num_indices - start;
  len = room <= 0 ? 0 : (int)min((long long)len, room);
}

// One bag per wavefront. OFF32: every row's byte offset fits 32 bits, so row
// addresses are formed as a uniform base plus a 32-bit per-lane offset.
template <int BPL, bool IS4, bool SO16, bool ACC16, bool OFF32>
__global__ __launch_bounds__(kSlwsThreads) void slws_wave_kernel(SlwsArgs a) {
  select_table(a);
  constexpr int kGroups = kSlwsThreads / 64;
  constexpr int kColsPerByte = IS4 ? 2 : 1;
  constexpr int kColsPerLane = BPL * kColsPerByte;
  constexpr int kGroup = 4;   // lookups handled under one uniform branch
  __shared__ long long s_part[kGroups];
  __shared__ __attribute__((aligned(16))) int s_own[kGroups];
  // per wave, per lookup of the batch: {row offset or row, weight, scale, offset}
  __shared__ int4 s_look[kGroups][kBatch];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const long long first_bag = (long long)blockIdx.x * kGroups;
  const long long bag = first_bag + wave;

  long long start;
  int len;
  wave_bag_span(a, tid, wave, bag, first_bag, s_part, s_own, start, len);
  int4 *look = s_look[wave];

  const int n_passes = (a.data_bytes + 64 * BPL - 1) / (64 * BPL);
  for (int pass = 0; pass < n_passes; pass++) {
    const int byte0 = (pass * 64 + lane) * BPL;
    const bool lane_live = byte0 < a.data_bytes;
    // lanes past the end of the row read its first bytes and store nothing
    const uint32_t lane_off = lane_live ? (uint32_t)byte0 : 0u;
    float acc[kColsPerLane];
#pragma unroll
    for (int c = 0; c < kColsPerLane; c++) acc[c] = 0.0f;

    for (int base = 0; base < len; base += kBatch) {
      const int cnt = min(kBatch, len - base);
      // first pass: lane j fetches lookup j of the batch
      int my_key;
      uint32_t so_lo = 0, so_hi = 0;
      float my_w;
      bool my_valid;
      {
        const long long pos = start + base + lane;
        long long row = -1;
        float w = 0.0f;
        if (lane < cnt && pos < a.num_indices) {
          row = a.idx64 ? reinterpret_cast<const long long *>(a.indices)[pos]
                        : (long long)reinterpret_cast<const int *>(a.indices)[pos];
          if (!a.weights) {
            w = 1.0f;
          } else if (a.w16) {
            w = __half2float(reinterpret_cast<const __half *>(a.weights)[pos]);
          } else {
            w = reinterpret_cast<const float *>(a.weights)[pos];
          }
        }
        // a skipped lookup reads row 0 and contributes w * 0
        my_valid = row >= 0 && row < a.data_rows;
        if (!my_valid) {
          row = 0;
          w = 0.0f;
        }
        my_w = w;
        my_key = OFF32 ? (int)(uint32_t)(row * a.in_line) : (int)row;
        // The row's scale and offset are requested here and consumed only
        // after the row reads below have been issued, so that the two
        // dependent round trips (index -> scale/offset, index -> row bytes)
        // overlap instead of following each other.
        if (!SO16 && a.sep_scales) {
          so_lo = __float_as_uint(a.sep_scales[row]);
          so_hi = __float_as_uint(a.sep_offsets[row]);
        } else {
          const uint8_t *so = a.data + row * a.in_line + a.data_bytes;
          so_lo = load_u32_any(so);
          if constexpr (!SO16) so_hi = load_u32_any(so + 4);
        }
      }
      // second pass: all row reads of the batch in flight before the first use.
      // Lookups are taken four at a time under one uniform branch; slots
      // beyond cnt hold {row 0, w 0, scale 0, offset 0} and add exactly +0.
      uint32_t q[kBatch];
#pragma unroll
      for (int g = 0; g < kBatch / kGroup; g++) {
        if (g * kGroup < cnt) {
          // An opaque copy of the 32-bit lane offset keeps its widening next
          // to the loads, which lets them use the scalar-base + 32-bit
          // vector-offset addressing form (global address space).
          uint32_t off = lane_off;
          asm volatile("" : "+v"(off));
#pragma unroll
          for (int u = 0; u < kGroup; u++) {
            const int j = g * kGroup + u;
            const int key = __builtin_amdgcn_readlane(my_key, j);
            // uniform row base (kept in scalar registers) + per-lane offset
            const uint8_t *rowp;
            if constexpr (OFF32) {
              rowp = a.data + (uint32_t)key;
            } else {
              rowp = a.data + (long long)key * a.in_line;
            }
            asm volatile("" : "+s"(rowp));
            const global_u8 *p = (const global_u8 *)rowp + off;
            if constexpr (BPL == 2) {
              q[j] = *(const global_u16 *)p;
            } else {
              q[j] = *p;
            }
          }
        }
      }
      {
        float s, o;
        if constexpr (SO16) {
          s = __half2float(__ushort_as_half((unsigned short)(so_lo & 0xffff)));
          o = __half2float(__ushort_as_half((unsigned short)(so_lo >> 16)));
        } else {
          s = __uint_as_float(so_lo);
          o = __uint_as_float(so_hi);
        }
        if (!my_valid) s = o = 0.0f;
        look[lane] = make_int4(my_key, __float_as_int(my_w), __float_as_int(s),
                               __float_as_int(o));
      }
      wave_lds_sync();
#pragma unroll
      for (int g = 0; g < kBatch / kGroup; g++) {
        if (g * kGroup < cnt) {
          int4 r[kGroup];
#pragma unroll
          for (int u = 0; u < kGroup; u++) r[u] = look[g * kGroup + u];
#pragma unroll
          for (int u = 0; u < kGroup; u++) {
            const int j = g * kGroup + u;
            const float w = __int_as_float(r[u].y), s = __int_as_float(r[u].z),
                        o = __int_as_float(r[u].w);
#pragma unroll
            for (int b = 0; b < BPL; b++) {
              const uint32_t byte = (q[j] >> (8 * b)) & 0xff;
              if constexpr (IS4) {
                acc[2 * b] = accumulate<ACC16>(acc[2 * b], w, s, o, byte & 15);
                acc[2 * b + 1] = accumulate<ACC16>(acc[2 * b + 1], w, s, o, byte >> 4);
              } else {
                acc[b] = accumulate<ACC16>(acc[b], w, s, o, byte);
              }
            }
          }
        }
      }
      wave_lds_sync(); // slots are rewritten by the next batch
    }

    if (bag < a.segments && lane_live)
      store_columns<kColsPerLane>(a, bag, byte0 * kColsPerByte, acc);
  }
}


// ---- fused-arithmetic variants ---------------------------------------------------
//
// Same operator with fused multiply-adds, for rows of 32 to 256 data
// bytes with fp32 accumulation.
//
// kMathElement (the default):
//   v = fma(s_j, q_jk, o_j);  dest[k] = fma(w_j, v, dest[k])
// the CPU loop's own expression w*(s*q+o) per element, with the two roundings
// of its products left out: three vector instructions per element (convert,
// fma, fma) instead of five. Each term differs from the CPU loop's by at most
// half a unit in the last place of s*q and of w*v, and nothing is regrouped,
// so a sum that cancels cancels here exactly where it does on the CPU.
//
// kMathRegrouped (on request only):
//   dest[k] = sum_j (w_j*s_j) * q_jk  +  sum_j (w_j*o_j)
// two instructions per element, but the two partial sums are large and of
// opposite sign for tables with a negative offset, so the error is relative to
// the magnitude a bag adds up and not to the result.
//
// One bag per wavefront; a lane reads 4 consecutive data bytes, so a row takes
// LPR = data_bytes/4 lanes and one load instruction fetches 64/LPR rows. The
// partial sums of the row groups are added across lanes at the end of the bag.
constexpr int kMathStrict = MI355X_SLWS_MATH_STRICT, kMathElement = MI355X_SLWS_MATH_ELEMENT,
              kMathRegrouped = MI355X_SLWS_MATH_REGROUPED;

// Cut points of the measurement entry point mi355x_frwq_slws_probe: the kernel
// stops after the named stage and stores a value that depends on what it read.
constexpr int kProbeOff = 0, kProbeSpan = 1, kProbeIndex = 2, kProbeScaleOffset = 3,
              kProbeRows = 4;

template <int MATH>
__device__ __forceinline__ float fused_term(const float4 &f, float q, float acc) {
  if constexpr (MATH == kMathElement) {
    return __fmaf_rn(f.x, __fmaf_rn(f.y, q, f.z), acc);   // f = {w, s, o}
  } else if constexpr (MATH == kMathStrict) {
    return __fadd_rn(acc, __fmul_rn(__fadd_rn(__fmul_rn(f.y, q), f.z), f.x));
  } else {
    return __fmaf_rn(f.x, q, acc);                        // f = {w*s, w*o}
  }
}

// (at any address)
typedef int __attribute__((ext_vector_type(4), aligned(1))) i32x4_any;
typedef uint32_t __attribute__((aligned(1))) u32_any;
typedef uint16_t __attribute__((aligned(1))) u16_any;
typedef i32x4_any __attribute__((address_space(1))) global_i32x4_any;
typedef u32_any __attribute__((address_space(1))) global_u32_any;
typedef u16_any __attribute__((address_space(1))) global_u16_any;
typedef uint32_t __attribute__((address_space(1))) global_u32;
typedef int32_t __attribute__((address_space(1))) global_i32;
typedef long long __attribute__((address_space(1))) global_i64;

// Sum of v over each row of 16 lanes, left in all 16 lanes of the row.
__device__ __forceinline__ uint32_t row16_sum_u32(uint32_t v) {
  int x = (int)v;
  x += __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xf, 0xf, true);  // quad_perm [1,0,3,2]
  x += __builtin_amdgcn_update_dpp(0, x, 0x4E, 0xf, 0xf, true);  // quad_perm [2,3,0,1]
  x += __builtin_amdgcn_update_dpp(0, x, 0x141, 0xf, 0xf, true); // row_half_mirror
  x += __builtin_amdgcn_update_dpp(0, x, 0x140, 0xf, 0xf, true); // row_mirror
  return (uint32_t)x;
}

// Span of the bag of wavefront `wave` of a block of WAVES wavefronts (WAVES
// consecutive bags per block), wave-uniform. Lengths mode: the block sums the
// clamped lengths in front of it (from the start of its chunk of
// bags, one 16-byte load per thread and trip, trips beyond the block's position
// skipped), one barrier, then lane g of every wave takes wave g's partial sum
// and bag g's length and a 16-lane sum gives the wave its start. The whole of
// it is about fifty vector instructions: with four waves on a SIMD every
// instruction a wave issues costs the launch sixteen cycles.
template <int WAVES>
__device__ __forceinline__ void rows_bag_span(const SlwsArgs &a, int tid, int lane, int wave,
                                              long long first_bag, uint32_t *s_part,
                                              long long *s_below, int *s_own,
                                              long long &start, int &len) {
  static_assert(WAVES % 4 == 0 && WAVES <= 16, "4, 8, 12 or 16 waves per block");
  constexpr int T = WAVES * 64;
  const long long bag = first_bag + wave;
  if (a.offsets) {
    long long start_v;
    int len_v;
    bag_span_offsets(a, bag, start_v, len_v);
    len = __builtin_amdgcn_readfirstlane(len_v);
    start = ((long long)__builtin_amdgcn_readfirstlane((int)(start_v >> 32)) << 32) |
            (unsigned int)__builtin_amdgcn_readfirstlane((int)start_v);
  } else {
    const long long chunk = a.chunk_sums ? first_bag / kChunkBags : 0;
    const long long lo = chunk * kChunkBags;
    const int32_t *lbase = a.lengths + lo;
    const int n_before = (int)(first_bag - lo);   // < kOneChunkBags, a multiple of WAVES
    const bool narrow = narrow_list(a);
    if (narrow) {
      const uint32_t part = wave_before<T>(lbase, n_before, a.chunk_sums, (int)chunk, tid,
                                           (int)a.num_indices);
      if (lane == 0) s_part[wave] = part;
    } else {
      const long long part = wave_before_wide<T>(lbase, n_before, a.chunk_sums, (int)chunk, tid);
      if (lane == 0) s_below[wave] = part;
    }
    if (tid < WAVES) {
      const long long b = first_bag + tid;
      s_own[tid] = (int)clamp_len(b < a.segments ? a.lengths[b] : 0,
                                  narrow ? (int)a.num_indices : 0x7fffffff);
    }
    __syncthreads();
    const int own = lane < WAVES ? s_own[lane] : 0;
    if (narrow) {
      const uint32_t p = lane < WAVES ? s_part[lane] : 0u;
      const uint32_t before = row16_sum_u32(p + (lane < wave ? (uint32_t)own : 0u));
      start = (long long)(uint32_t)__builtin_amdgcn_readlane((int)before, 0);
    } else {
      long long before = 0;
      for (int g = 0; g < WAVES; g++) before += s_below[g] + (g < wave ? s_own[g] : 0);
      start = ((long long)__builtin_amdgcn_readfirstlane((int)(before >> 32)) << 32) |
              (unsigned int)__builtin_amdgcn_readfirstlane((int)before);
    }
    len = bag < a.segments ? __builtin_amdgcn_readlane(own, wave) : 0;
  }
  const long long room = a.num_indices - start;
  len = room <= 0 ? 0 : (int)min((long long)len, room);
}

// Lookup j of a batch, in lane j: a skipped one (or none) has row 0 and is not valid.
struct Lookup {
  uint32_t row = 0;
  float w = 0.0f;
  bool valid = false;
};

// Lookups at .. at + cnt of the lists (uniform). The span never reaches past the index
// list, so lane < cnt is the only check. (Loads through global-address pointers: a
// generic-address load also counts as an LDS operation, and the wait for the keys of a
// batch would then wait for it.)
__device__ __forceinline__ Lookup fetch_lookup(const SlwsArgs &a, long long at, int cnt, int lane) {
  Lookup l;
  if (lane < cnt) {
    if (a.idx64) {
      const long long r = ((const global_i64 *)a.indices + at)[lane];
      l.valid = (unsigned long long)r < (unsigned long long)a.data_rows;
      l.row = (uint32_t)r;
    } else {
      l.row = (uint32_t)((const global_i32 *)a.indices + at)[lane];
      l.valid = l.row < (uint32_t)a.data_rows;
    }
    if (!a.weights) {
      l.w = 1.0f;
    } else if (a.w16) {
      l.w = __half2float(__ushort_as_half(((const global_u16 *)a.weights + at)[lane]));
    } else {
      l.w = __uint_as_float(((const global_u32 *)a.weights + at)[lane]);
    }
  }
  if (!l.valid) l.row = 0;
  return l;
}

// The same in two halves for a wavefront that asks for its lookups a batch ahead: index and
// weight as they lie in their lists (all ones for a lane without a lookup; `hi` only of
// 64-bit indices), not waited for. The two parts of an address are pinned where they are:
// in a loop the compiler otherwise keeps one sum of base and lane per list and type,
// sixteen vector registers.
struct RawLookup {
  uint32_t lo = ~0u, hi = ~0u, w = 0;
};
__device__ __forceinline__ RawLookup request_lookup(const SlwsArgs &a, long long at, int cnt, int lane) {
  RawLookup r;
  auto from = [&](const void *list, int bytes) {
    const global_u8 *p = (const global_u8 *)list + at * bytes;
    uint32_t off = (uint32_t)(lane * bytes);
    asm("" : "+s"(p), "+v"(off));
    return p + off;
  };
  if (lane < cnt) {
    if (a.idx64) {
      const long long v = *(const global_i64 *)from(a.indices, 8);
      r.lo = (uint32_t)v;
      r.hi = (uint32_t)((unsigned long long)v >> 32);
    } else {
      r.lo = (uint32_t)*(const global_i32 *)from(a.indices, 4);
    }
    if (a.weights)
      r.w = a.w16 ? (uint32_t)*(const global_u16 *)from(a.weights, 2)
                  : *(const global_u32 *)from(a.weights, 4);
  }
  return r;
}
__device__ __forceinline__ Lookup settle_lookup(const SlwsArgs &a, const RawLookup &r) {
  Lookup l;
  l.valid = r.lo < (uint32_t)a.data_rows && (!a.idx64 || r.hi == 0);   // data_rows < 2^31
  l.row = l.valid ? r.lo : 0u;
  l.w = !a.weights ? 1.0f
        : a.w16    ? __half2float(__ushort_as_half((unsigned short)r.w))
                   : __uint_as_float(r.w);
  return l;
}

// A bag's running sums in one wavefront, rows of up to LPR * 4 data bytes (a multiple of 4
// and 4-byte aligned rows; lanes past a narrower row read its first word and store
// nothing). ANY = 1, 2 or 4: rows of any width from that on, at any address, as many bytes
// to a lane, the last lane the ones that end the row.
template <bool IS4, bool SO16, int LPR, bool OFF32, int MATH, int PROBE = kProbeOff, int ANY = 0,
          int ROUND = kBatch>
struct RowsBag {
  typedef typename std::conditional<ANY != 0, global_u32_any, global_u32>::type word;
  static constexpr int kBytes = ANY ? ANY : 4;   // of a row per lane
  static constexpr int RPI = 64 / LPR;           // rows per load instruction
  static constexpr int kCols = IS4 ? 2 * kBytes : kBytes; // output columns per lane
  static constexpr int kLoads = ROUND / RPI;     // load instructions of a full batch
  static constexpr int kChunk = kLoads < 4 ? kLoads : 4; // loads under one uniform branch

  int sub, lir;                           // which row of a load this lane reads, where in it
  bool live;
  uint32_t lane_off;
  float acc[kCols], acc_o;

  __device__ __forceinline__ RowsBag(const SlwsArgs &a, int lane)
      : sub(lane / LPR), lir(lane % LPR), live(lir * kBytes < a.data_bytes),
        lane_off(!live ? 0u : (uint32_t)(ANY ? min(lir * kBytes, a.data_bytes - kBytes) : lir * 4)) {
    clear();
  }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int c = 0; c < kCols; c++) acc[c] = 0.0f;
    acc_o = 0.0f;
  }

  // One batch of cnt <= ROUND lookups, lane j holding lookup j. keys and wso: kBatch entries
  // of the wavefront's own. `meanwhile` is called with the scales and offsets asked for and
  // no row yet.
  template <class F>
  __device__ __forceinline__ void batch(const SlwsArgs &a, const Lookup &my, int cnt, int lane,
                                        uint32_t *keys, float4 *wso, F meanwhile) {
    // first pass: lane j turns to lookup j. A skipped lookup reads row 0 and contributes
    // exactly +0.
    const uint32_t row = my.row;
    const bool sep = !SO16 && a.sep_scales != nullptr;   // uniform
    // The row's scale and offset are requested here and consumed only after
    // the row reads below have been issued, so that the two round trips that
    // depend on the index (scale/offset, row bytes) overlap.
    uint32_t so_lo = 0, so_hi = 0;
    if (sep) {
      so_lo = ((const global_u32 *)a.sep_scales)[row];
      so_hi = ((const global_u32 *)a.sep_offsets)[row];
    } else if constexpr (OFF32) {
      const uint32_t key = row * (uint32_t)a.in_line;
      const global_u8 *so = (const global_u8 *)a.data + a.data_bytes;
      so_lo = *(const word *)(so + key);
      if constexpr (!SO16) so_hi = *(const word *)(so + key + 4u);
    } else {
      const global_u32 *so = (const global_u32 *)((const global_u8 *)a.data +
                                                  ((long long)row * a.in_line + a.data_bytes));
      so_lo = so[0];
      if constexpr (!SO16) so_hi = so[1];
    }
    keys[lane] = OFF32 ? row * (uint32_t)a.in_line : row;
    if constexpr (PROBE == kProbeIndex) {
      // measurement only: up to the index and weight of every lookup
      acc_o += my.w + (float)row;
      return;
    }
    if constexpr (PROBE == kProbeScaleOffset) {
      // measurement only: up to the scale and offset of every lookup
      acc_o += my.valid ? my.w * __uint_as_float(so_lo) + __uint_as_float(so_hi) : 0.0f;
      return;
    }
    meanwhile();
    wave_lds_sync();
    // second pass: all row reads of the batch in flight before the first use,
    // kChunk load instructions per chunk, as many chunks as the batch has
    // lookups for. The chunk count is wave-uniform and picks one straight-line
    // body (loads of N chunks, the park of {w, s, o}, arithmetic of N chunks):
    // with the chunks under separate branches the loaded words become values
    // carried around the loop and cost a register copy each per batch. Slots
    // beyond cnt hold {row 0, 0, 0, 0} and add exactly +0.
    auto second_pass = [&](auto nc) {
      constexpr int N = decltype(nc)::value;   // chunks
      uint32_t q[N * kChunk];
#pragma unroll
      for (int g = 0; g < N * kChunk; g++) {
        const uint32_t key = keys[g * RPI + sub];
        if constexpr (ANY == 1) {
          q[g] = *((const global_u8 *)a.data + (key + lane_off));
        } else if constexpr (ANY == 2) {
          q[g] = *(const global_u16_any *)((const global_u8 *)a.data + (key + lane_off));
        } else if constexpr (OFF32) {
          q[g] = *(const word *)((const global_u8 *)a.data + (key + lane_off));
        } else {
          q[g] = *reinterpret_cast<const uint32_t *>(
              a.data + (long long)key * a.in_line + lane_off);
        }
      }
      // (no use of a row between the requests: its wait would hold back the rest)
      __builtin_amdgcn_sched_barrier(0);
      {
        float sc, of;
        if constexpr (SO16) {
          sc = __half2float(__ushort_as_half((unsigned short)(so_lo & 0xffff)));
          of = __half2float(__ushort_as_half((unsigned short)(so_lo >> 16)));
        } else {
          sc = __uint_as_float(so_lo);
          of = __uint_as_float(so_hi);
        }
        if constexpr (MATH != kMathRegrouped)
          wso[lane] = my.valid ? make_float4(my.w, sc, of, 0.0f)
                               : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        else
          wso[lane] = my.valid ? make_float4(my.w * sc, my.w * of, 0.0f, 0.0f)
                               : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      }
      wave_lds_sync();
#pragma unroll
      for (int g = 0; g < N * kChunk; g++) {
        if constexpr (PROBE == kProbeRows) {
          // measurement only: every row read, no arithmetic
          acc_o = __uint_as_float(__float_as_uint(acc_o) ^ q[g]);
          continue;
        }
        const float4 f = wso[g * RPI + sub];
        if constexpr (MATH == kMathRegrouped) acc_o += f.y;
        if constexpr (IS4) {
          const uint32_t lo = q[g] & 0x0f0f0f0fu, hi = (q[g] >> 4) & 0x0f0f0f0fu;
#pragma unroll
          for (int b = 0; b < kBytes; b++) {
            acc[2 * b] = fused_term<MATH>(f, (float)((lo >> (8 * b)) & 0xff), acc[2 * b]);
            acc[2 * b + 1] =
                fused_term<MATH>(f, (float)((hi >> (8 * b)) & 0xff), acc[2 * b + 1]);
          }
        } else {
#pragma unroll
          for (int b = 0; b < kBytes; b++)
            acc[b] = fused_term<MATH>(f, (float)((q[g] >> (8 * b)) & 0xff), acc[b]);
        }
      }
    };
    constexpr int kChunks = kLoads / kChunk;
    static_assert(kChunks <= 16, "one case per chunk count");
    const int chunks = (cnt + kChunk * RPI - 1) / (kChunk * RPI);   // 1..kChunks, uniform
#define MI355X_SECOND_PASS(n)                                                  \
  case n:                                                                      \
    if constexpr (n <= kChunks) second_pass(std::integral_constant<int, (n <= kChunks ? n : 1)>()); \
    break;
    switch (chunks) {
      MI355X_SECOND_PASS(1) MI355X_SECOND_PASS(2) MI355X_SECOND_PASS(3) MI355X_SECOND_PASS(4)
      MI355X_SECOND_PASS(5) MI355X_SECOND_PASS(6) MI355X_SECOND_PASS(7) MI355X_SECOND_PASS(8)
      MI355X_SECOND_PASS(9) MI355X_SECOND_PASS(10) MI355X_SECOND_PASS(11) MI355X_SECOND_PASS(12)
      MI355X_SECOND_PASS(13) MI355X_SECOND_PASS(14) MI355X_SECOND_PASS(15) MI355X_SECOND_PASS(16)
    default:
      break;
    }
#undef MI355X_SECOND_PASS
    wave_lds_sync(); // slots are rewritten by the next batch
  }

  // The bag's sums: partial sums of the RPI row groups -> lanes of group 0, stored.
  __device__ __forceinline__ void finish(const SlwsArgs &a, long long bag) {
    if constexpr (PROBE == kProbeRows) acc_o = (float)(__float_as_uint(acc_o) & 0xffu);
#pragma unroll
    for (int c = 0; c < kCols; c++) {
      float v = MATH == kMathRegrouped || PROBE != kProbeOff ? acc[c] + acc_o : acc[c];
#pragma unroll
      for (int off = LPR; off < 64; off <<= 1) v += __shfl_xor(v, off, 64);
      acc[c] = v;
    }
    if (bag < a.segments && sub == 0 && live)
      store_columns<kCols>(a, bag, ANY ? (int)lane_off * (IS4 ? 2 : 1) : lir * kCols, acc);
  }
};

// A whole bag by one wavefront (RowsBag), whose arguments are wave-uniform.
template <bool IS4, bool SO16, int LPR, bool OFF32, int MATH, int PROBE = kProbeOff, int ANY = 0>
__device__ __forceinline__ void rows_bag(const SlwsArgs &a, long long bag, long long start, int len,
                                         int lane, uint32_t *keys, float4 *wso) {
  if constexpr (PROBE == kProbeSpan) {
    // measurement only: the launch up to the bags' positions
    if (bag < a.segments && lane == 0)
      reinterpret_cast<float *>(a.dest)[bag * a.out_cols] = (float)(start + len);
    return;
  }
  RowsBag<IS4, SO16, LPR, OFF32, MATH, PROBE, ANY> sums(a, lane);
  for (int base = 0; base < len; base += kBatch) {
    const int cnt = min(kBatch, len - base);
    sums.batch(a, fetch_lookup(a, start + base, cnt, lane), cnt, lane, keys, wso, [] {});
  }
  sums.finish(a, bag);
}

// One bag per wavefront, WAVES bags per block (rows_bag). Eight-bit rows with fp32 scales take
// 64 registers (65 before), so that two blocks of sixteen wavefronts fit a CU: 128 columns
// 4096 x 40 7.7 -> 7.5 us and 8143 x 30 10.7 -> 9.2, inputs changing. (Held to 64 where it takes one more, rows of
// 128 columns, 4096 x 40, go 7.6 -> 7.9.)
template <bool IS4, bool SO16, int LPR, bool OFF32, int MATH, int WAVES,
          int PROBE = kProbeOff>
__global__ __launch_bounds__(WAVES * 64) void slws_rows_kernel(SlwsArgs a) {
  select_table(a);
  __shared__ uint32_t s_part[WAVES];
  __shared__ long long s_below[WAVES];
  __shared__ int s_own[WAVES];
  // per wave, per lookup of the batch: row byte offset (or row) and
  // {w, s, o} (kMathElement) or {w*s, w*o} (kMathRegrouped)
  __shared__ uint32_t s_key[WAVES][kBatch];
  __shared__ float4 s_ws[WAVES][kBatch];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long long first_bag = (long long)blockIdx.x * WAVES;

  long long start;
  int len;
  rows_bag_span<WAVES>(a, tid, lane, wave, first_bag, s_part, s_below, s_own, start, len);
  rows_bag<IS4, SO16, LPR, OFF32, MATH, PROBE>(a, first_bag + wave, start, len, lane, s_key[wave],
                                               s_ws[wave]);
}

// A range of `per_block` consecutive bags per block (at most 64), its wavefronts taking them
// one after the other as they come free. With a bag per wavefront a launch of many bags pays
// three dependent trips to memory (lengths, indices, rows) per bag and turn of the resident
// wavefronts; here the positions of a block's bags are formed once, and a wavefront asks for
// the lookups of its next batch, of the next bag as well, before it reads the rows of the
// batch in hand, so that a bag costs one trip, which the other wavefronts of the SIMD cover.
// What bounds it is then the rate of random 64-byte accesses behind L2 (some 65 G/s; 100
// columns 30 000 x 30, 84 MB from there, 20 us without the positions) or, where the table
// lies in L2, vector instructions (2489 rows of 200 columns, 55 288 x 13). The bags are dealt
// by an LDS counter: a long one holds up its wavefront and no other. Same bits as
// slws_rows_kernel (a column's parts and their order). A round of 64 lookups takes 32 row
// words a lane at 32 lanes to a row, 67 registers; at 64 lanes rounds of 32 keep it at seven
// wavefronts per SIMD instead of four (55 288 x 13 37 / 32 us). Forced to 64 registers it
// spills three and is slower (100 columns 30 000 x 30 26.3 / 28.7). us, slws_rows_kernel or
// slws_wide_kernel before / this one, lengths Poisson: 100 columns 30 000 x 30 29.8 / 25.9;
// 128 columns 6000 x 30 8.8 / 6.6, 13 000 x 15 13.3 / 9.9, 20 000 x 20 18.6 / 15.3, 65 000 x
// 39 60.6 / 53, 150 000 x 12 90 / 61; 200 columns 2489 rows 55 288 x 13 51.1 / 32.1, 30 000 x
// 8 23.6 / 17.7; 256 columns 9558 x 25 16.8 / 13.7, 5000 x 30 11.8 / 9.0; 200 and 256 columns
// of four bits 30 000 x 30 35.9 / 33.3, 14 000 x 40 26.7 / 20.5 (from 16 385 to kRangesOneBags bags
// with the launch that sums chunks in front; 1 to 2 us less without it).
template <bool IS4, bool SO16, int LPR, bool OFF32, int MATH, int WAVES, int ROUND>
__global__ __launch_bounds__(WAVES * 64) void slws_ranges_kernel(SlwsArgs a, int per_block) {
  constexpr int T = WAVES * 64;
  __shared__ long long s_before[WAVES];
  __shared__ int s_next;
  __shared__ long long s_start[64];
  __shared__ int s_len[64];
  __shared__ uint32_t s_key[WAVES][64];
  __shared__ float4 s_ws[WAVES][64];

  a.out_q8 = 0;                        // (multi-table launches only)
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long long first_bag = (long long)blockIdx.x * per_block;
  const int bags = (int)min((long long)per_block, a.segments - first_bag);
  {
    // lane g of the first wavefront: where bag g of the block starts, its lookups
    long long start = 0;
    int len = 0;
    if (a.offsets) {
      if (wave == 0 && lane < bags) bag_span_offsets(a, first_bag + lane, start, len);
    } else {
      const long long chunk = a.chunk_sums ? first_bag / kChunkBags : 0;
      const long long lo = chunk * kChunkBags;
      const int32_t *lbase = a.lengths + lo;
      const int n_before = (int)(first_bag - lo);   // < kRangesOneBags, a multiple of 4
      const int own = tid < bags ? a.lengths[first_bag + tid] : 0;
      if (narrow_list(a)) {
        const int most = (int)a.num_indices;
        const uint32_t part =
            a.chunk_sums ? wave_before<T>(lbase, n_before, a.chunk_sums, (int)chunk, tid, most)
                         : wave_before_long<T>(lbase, n_before, tid, most);
        if (lane == 0) s_before[wave] = part;
        __syncthreads();
        if (wave == 0) {
          uint32_t before = 0;                       // eight sums below 2^26
#pragma unroll
          for (int w = 0; w < WAVES; w++) before += (uint32_t)s_before[w];
          // 64 lengths below 2^26 stay inside 32 bits
          const uint32_t cut = clamp_len(own, most);
          start = (long long)before + (wave_scan_u32(cut) - cut);
          len = (int)cut;
        }
      } else {
        const long long part = wave_before_wide<T>(lbase, n_before, a.chunk_sums, (int)chunk, tid);
        if (lane == 0) s_before[wave] = part;
        __syncthreads();
        if (wave == 0) {
          len = (int)clamp_len(own);
          long long scan = len;
#pragma unroll
          for (int off = 1; off < 64; off <<= 1) {
            const long long v = __shfl_up(scan, off, 64);
            if (lane >= off) scan += v;
          }
          start = scan - len;
          for (int w = 0; w < WAVES; w++) start += s_before[w];
        }
      }
      const long long room = a.num_indices - start;
      len = room <= 0 ? 0 : (int)min((long long)len, room);
    }
    if (wave == 0) {
      s_start[lane] = start;
      s_len[lane] = len;
      if (lane == 0) s_next = WAVES;
    }
    __syncthreads();
  }

  RowsBag<IS4, SO16, LPR, OFF32, MATH, kProbeOff, 0, ROUND> sums(a, lane);
  // the bag in hand, its first lookups asked for
  int bag = wave, len = 0;
  long long start = 0;
  auto turn_to = [&](int g) {
    bag = g;
    len = 0;
    if (g < bags) {
      len = __builtin_amdgcn_readfirstlane(s_len[g]);
      const long long at = s_start[g];
      start = ((long long)__builtin_amdgcn_readfirstlane((int)(at >> 32)) << 32) |
              (unsigned int)__builtin_amdgcn_readfirstlane((int)at);
    }
  };
  turn_to(wave);
  RawLookup raw = request_lookup(a, start, min(ROUND, len), lane);
  __builtin_amdgcn_s_waitcnt(0x0f70);                // vmcnt(0): see below
  while (bag < bags) {
    int next = 0;
    if (lane == 0) next = atomicAdd(&s_next, 1);
    next = __builtin_amdgcn_readfirstlane(next);
    const long long mine = first_bag + bag;
    const int my_len = len;
    const long long my_start = start;
    turn_to(next);
    sums.clear();
    int base = 0;
    do {
      const int cnt = min(ROUND, my_len - base);
      const RawLookup now = raw;
      base += ROUND;
      const bool more = base < my_len;
      // the lookups behind these: of the bag, or the first ones of the next
      auto ahead = [&] {
        raw = request_lookup(a, more ? my_start + base : start, min(ROUND, more ? my_len - base : len), lane);
      };
      if (cnt > 0) {
        sums.batch(a, settle_lookup(a, now), cnt, lane, s_key[wave], s_ws[wave], ahead);
      } else {
        // waited for here (the rows' waits cover it in the other branch), so that no
        // lookup is on its way at the loop's head, where its wait would be for the
        // stores of the bag before too
        ahead();
        __builtin_amdgcn_s_waitcnt(0x0f70);          // vmcnt(0)
      }
    } while (base < my_len);
    sums.finish(a, mine);
  }
}

// The same operator for short rows (up to 64 data bytes, a multiple of 4): a row
// takes only LPR = 4, 8 or 16 lanes, so a wavefront works on 64/LPR bags side by
// side, one per lane group, and nothing has to be added across lanes at the end.
// A group's lanes fetch its lookups (index, weight, scale, offset) kGB at a
// time and hand them to each other through a wave-private LDS table. A lane adds
// its columns up in bag order, so the strict arithmetic runs here as well; there
// rows of less than 32 bytes may also run with BPL = 1 data byte per lane, which
// shortens a lane's chain of dependent operations to a quarter.
template <bool IS4, bool SO16, int LPR, bool OFF32, int MATH, int BPL = 4>
__global__ __launch_bounds__(kSlwsThreads) void slws_groups_kernel(SlwsArgs a) {
  select_table(a);
  constexpr int kGroups = kSlwsThreads / LPR; // bags per block
  constexpr int kCols = (IS4 ? 2 : 1) * BPL;  // output columns per lane
  constexpr int kGB = 32;                     // lookups of a bag per round
  constexpr int kPer = kGB / LPR;             // lookups one lane fetches per round
  constexpr int kChunk = 8;                   // row reads under one uniform branch
  __shared__ long long s_part[kSlwsThreads / 64];
  __shared__ int s_own[kGroups];
  // one entry of padding per bag: the bags of a wavefront read the same slot of
  // their own tables at once, which lie in different banks that way
  __shared__ uint32_t s_key[kGroups][kGB + 1];
  __shared__ float4 s_ws[kGroups][kGB + 1];

  const int tid = threadIdx.x;
  const int grp = tid / LPR, lir = tid % LPR;
  const long long first_bag = (long long)blockIdx.x * kGroups;
  const long long bag = first_bag + grp;

  long long start = 0;
  int len = 0;
  bag_span<kGroups>(a, tid, grp, bag, first_bag, s_part, s_own, start, len);
  {
    const long long room = a.num_indices - start;
    len = room <= 0 ? 0 : (int)min((long long)len, room);
  }
  // the loops below run as long as the longest bag of the wavefront needs
  int wave_len = len;
#pragma unroll
  for (int off = LPR; off < 64; off <<= 1) wave_len = max(wave_len, __shfl_xor(wave_len, off, 64));
  wave_len = __builtin_amdgcn_readfirstlane(wave_len);

  uint32_t *keys = s_key[grp];
  float4 *wso = s_ws[grp];
  const bool live = lir * BPL < a.data_bytes;
  const uint32_t lane_off = live ? (uint32_t)(lir * BPL) : 0u;
  float acc[kCols];
  float acc_o = 0.0f;
#pragma unroll
  for (int c = 0; c < kCols; c++) acc[c] = 0.0f;

  for (int base = 0; base < wave_len; base += kGB) {
    const int cnt = min(kGB, len - base);           // this bag's share (may be <= 0)
    const int wave_cnt = min(kGB, wave_len - base); // uniform
    // scale and offset are requested with the index in hand and consumed after
    // the row reads have been issued (global-address loads: see slws_rows_kernel)
    uint32_t so_lo[kPer], so_hi[kPer];
    float my_w[kPer];
    bool my_valid[kPer];
#pragma unroll
    for (int k = 0; k < kPer; k++) {
      const int j = lir + k * LPR;
      const long long pos = start + base + j;
      long long row = -1;
      float w = 0.0f;
      if (j < cnt && pos < a.num_indices) {
        row = a.idx64 ? ((const global_i64 *)a.indices)[pos]
                      : (long long)((const global_i32 *)a.indices)[pos];
        if (!a.weights) {
          w = 1.0f;
        } else if (a.w16) {
          w = __half2float(reinterpret_cast<const __half *>(a.weights)[pos]);
        } else {
          w = reinterpret_cast<const float *>(a.weights)[pos];
        }
      }
      // a skipped lookup reads row 0 and contributes exactly +0
      my_valid[k] = row >= 0 && row < a.data_rows;
      if (!my_valid[k]) row = 0;
      my_w[k] = w;
      so_hi[k] = 0;
      if (!SO16 && a.sep_scales) {
        so_lo[k] = ((const global_u32 *)a.sep_scales)[row];
        so_hi[k] = ((const global_u32 *)a.sep_offsets)[row];
      } else {
        const global_u32 *so = (const global_u32 *)((const global_u8 *)a.data +
                                                    (row * a.in_line + a.data_bytes));
        so_lo[k] = so[0];
        if constexpr (!SO16) so_hi[k] = so[1];
      }
      keys[j] = OFF32 ? (uint32_t)(row * a.in_line) : (uint32_t)row;
    }
    wave_lds_sync();
    uint32_t q[kGB];
#pragma unroll
    for (int c = 0; c < kGB / kChunk; c++) {
      if (c * kChunk < wave_cnt) {
#pragma unroll
        for (int u = 0; u < kChunk; u++) {
          const int j = c * kChunk + u;
          const uint32_t key = keys[j];
          if constexpr (BPL == 1) {
            q[j] = *((const global_u8 *)a.data +
                     (OFF32 ? (unsigned long long)key : (unsigned long long)key * a.in_line) +
                     lane_off);
          } else if constexpr (OFF32) {
            q[j] = *(const global_u32 *)((const global_u8 *)a.data + (key + lane_off));
          } else {
            q[j] = *reinterpret_cast<const uint32_t *>(
                a.data + (long long)key * a.in_line + lane_off);
          }
        }
      }
    }
#pragma unroll
    for (int k = 0; k < kPer; k++) {
      float sc, of;
      if constexpr (SO16) {
        sc = __half2float(__ushort_as_half((unsigned short)(so_lo[k] & 0xffff)));
        of = __half2float(__ushort_as_half((unsigned short)(so_lo[k] >> 16)));
      } else {
        sc = __uint_as_float(so_lo[k]);
        of = __uint_as_float(so_hi[k]);
      }
      if constexpr (MATH != kMathRegrouped)
        wso[lir + k * LPR] = my_valid[k] ? make_float4(my_w[k], sc, of, 0.0f)
                                         : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      else
        wso[lir + k * LPR] = my_valid[k] ? make_float4(my_w[k] * sc, my_w[k] * of, 0.0f, 0.0f)
                                         : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    wave_lds_sync();
#pragma unroll
    for (int c = 0; c < kGB / kChunk; c++) {
      if (c * kChunk < wave_cnt) {
#pragma unroll
        for (int u = 0; u < kChunk; u++) {
          const int j = c * kChunk + u;
          const float4 f = wso[j];
          if constexpr (MATH == kMathRegrouped) acc_o += f.y;
          if constexpr (IS4) {
            const uint32_t lo = q[j] & 0x0f0f0f0fu, hi = (q[j] >> 4) & 0x0f0f0f0fu;
#pragma unroll
            for (int b = 0; b < BPL; b++) {
              acc[2 * b] = fused_term<MATH>(f, (float)((lo >> (8 * b)) & 0xff), acc[2 * b]);
              acc[2 * b + 1] =
                  fused_term<MATH>(f, (float)((hi >> (8 * b)) & 0xff), acc[2 * b + 1]);
            }
          } else {
#pragma unroll
            for (int b = 0; b < BPL; b++)
              acc[b] = fused_term<MATH>(f, (float)((q[j] >> (8 * b)) & 0xff), acc[b]);
          }
        }
      }
    }
    wave_lds_sync(); // slots are rewritten by the next round
  }
#pragma unroll
  for (int c = 0; c < kCols; c++)
    if constexpr (MATH == kMathRegrouped) acc[c] += acc_o;
  if (bag < a.segments && live) store_columns<kCols>(a, bag, lir * kCols, acc);
}

// The same operator for many short bags of eight-bit rows, of 65 to 128 bytes that start on a
// word or of 33 to 256 at any address, bound by what a bag costs beside its rows: a lane reads sixteen bytes of a row, so that
// LPR = 4, 8 or 16 lanes hold one and a wavefront works on the rows of several bags at once,
// side by side as in slws_groups_kernel. PARTS = 2: a bag's even and odd lookups go to two
// groups of lanes and are added at the end, which is the order in which slws_rows_kernel sums
// rows of 65 to 128 bytes; 1: in bag order. The last lane of a row reads the sixteen bytes that
// end with it; columns that two lanes hold are the same values and stored twice.
template <bool SO16, int LPR, int PARTS, int MATH>
__global__ __launch_bounds__(kSlwsThreads) void slws_wide_kernel(SlwsArgs a) {
  select_table(a);
  constexpr int kLanes = LPR * PARTS;            // of a bag
  constexpr int kGroups = kSlwsThreads / kLanes; // bags per block
  constexpr int kCols = 16;                      // output columns per lane
  constexpr int kPer = 4;                        // lookups one lane fetches per round
  constexpr int kGB = kLanes * kPer;             // lookups of a bag per round
  // row reads of a lane in flight (eight: forty registers more, two waves per SIMD fewer and
  // a bag's last step half empty, 3 to 30 % slower)
  constexpr int kRows = 4;
  constexpr int kStep = kRows * PARTS;
  static_assert(kGB % kStep == 0, "whole steps per round");
  __shared__ long long s_part[kSlwsThreads / 64];
  __shared__ int s_own[kGroups];
  __shared__ int s_longs;             // how many bags go to a wavefront of their own: which
  __shared__ int4 s_long[kGroups];
  // (an entry of padding per bag: see slws_groups_kernel)
  __shared__ uint32_t s_key[kGroups][kGB + 1];
  __shared__ float4 s_ws[kGroups][kGB + 1];

  const int tid = threadIdx.x;
  const int grp = tid / kLanes, lib = tid % kLanes;
  const int part = lib / LPR, lir = lib % LPR;
  const long long first_bag = (long long)blockIdx.x * kGroups;
  const long long bag = first_bag + grp;

  if (tid == 0) s_longs = 0;
  long long start = 0;
  int len = 0;
  bag_span<kGroups>(a, tid, grp, bag, first_bag, s_part, s_own, start, len);
  {
    const long long room = a.num_indices - start;
    len = room <= 0 ? 0 : (int)min((long long)len, room);
  }
  // A bag much longer than the launch's average goes to a whole wavefront, the block's long
  // bags in turn to its waves: beside the others it would go on eight lookups at a time.
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool alone = len > a.long_bag;
  __syncthreads();
  if (alone && lib == 0)
    s_long[atomicAdd(&s_longs, 1)] = make_int4((int)start, (int)(start >> 32), len, grp);
  __syncthreads();
  for (int i = wave; i < s_longs; i += kSlwsThreads / 64) {
    const int4 b = s_long[i];
    const long long first = ((long long)__builtin_amdgcn_readfirstlane(b.y) << 32) |
                            (unsigned int)__builtin_amdgcn_readfirstlane(b.x);
    rows_bag<false, SO16, 64 / PARTS, true, MATH, kProbeOff, MATH == kMathStrict ? LPR / 4 : 0>(
        a, first_bag + __builtin_amdgcn_readfirstlane(b.w), first,
        __builtin_amdgcn_readfirstlane(b.z), lane, s_key[wave * (64 / kLanes)],
        s_ws[wave * (64 / kLanes)]);
  }
  if (alone) len = 0;
  // the loops below run as long as the longest bag of the wavefront needs
  int wave_len = len;
#pragma unroll
  for (int off = kLanes; off < 64; off <<= 1) wave_len = max(wave_len, __shfl_xor(wave_len, off, 64));
  wave_len = __builtin_amdgcn_readfirstlane(wave_len);

  uint32_t *keys = s_key[grp];
  float4 *wso = s_ws[grp];
  const bool live = lir * 16 < a.data_bytes;
  const uint32_t lane_off = live ? (uint32_t)min(lir * 16, a.data_bytes - 16) : 0u;
  const global_u8 *data = (const global_u8 *)a.data;
  float acc[kCols];
#pragma unroll
  for (int c = 0; c < kCols; c++) acc[c] = 0.0f;

  for (int base = 0; base < wave_len; base += kGB) {
    const int cnt = min(kGB, len - base);           // this bag's share (may be <= 0)
    // slots that the steps below read, uniform
    const int wave_cnt = (min(kGB, wave_len - base) + kStep - 1) / kStep * kStep;
    uint32_t so_lo[kPer], so_hi[kPer];
    float my_w[kPer];
    bool my_valid[kPer];
#pragma unroll
    for (int k = 0; k < kPer; k++) {
      so_lo[k] = so_hi[k] = 0;
      my_w[k] = 0.0f;
      my_valid[k] = false;
      if (k * kLanes < wave_cnt) {
        const int j = lib + k * kLanes;
        const long long pos = start + base + j;
        long long row = -1;
        if (j < cnt) {
          row = a.idx64 ? ((const global_i64 *)a.indices)[pos]
                        : (long long)((const global_i32 *)a.indices)[pos];
          if (!a.weights) my_w[k] = 1.0f;
          else if (a.w16) my_w[k] = __half2float(__ushort_as_half(((const global_u16 *)a.weights)[pos]));
          else my_w[k] = __uint_as_float(((const global_u32 *)a.weights)[pos]);
        }
        // a skipped lookup reads row 0 and contributes exactly +0
        my_valid[k] = row >= 0 && row < a.data_rows;
        if (!my_valid[k]) row = 0;
        if (!SO16 && a.sep_scales) {
          so_lo[k] = ((const global_u32 *)a.sep_scales)[row];
          so_hi[k] = ((const global_u32 *)a.sep_offsets)[row];
        } else {
          const global_u32_any *so =
              (const global_u32_any *)(data + ((uint32_t)row * (uint32_t)a.in_line + (uint32_t)a.data_bytes));
          so_lo[k] = so[0];
          if constexpr (!SO16) so_hi[k] = so[1];
        }
        keys[j] = (uint32_t)row * (uint32_t)a.in_line;
      }
    }
    wave_lds_sync();
    i32x4 q[kRows];
    auto request = [&](int c) {
#pragma unroll
      for (int u = 0; u < kRows; u++)
        q[u] = *(const global_i32x4_any *)(data + (keys[c + u * PARTS + part] + lane_off));
    };
    request(0);
#pragma unroll
    for (int k = 0; k < kPer; k++) {
      if (k * kLanes < wave_cnt) {
        float sc, of;
        if constexpr (SO16) {
          sc = __half2float(__ushort_as_half((unsigned short)(so_lo[k] & 0xffff)));
          of = __half2float(__ushort_as_half((unsigned short)(so_lo[k] >> 16)));
        } else {
          sc = __uint_as_float(so_lo[k]);
          of = __uint_as_float(so_hi[k]);
        }
        wso[lib + k * kLanes] = my_valid[k] ? make_float4(my_w[k], sc, of, 0.0f)
                                            : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      }
    }
    wave_lds_sync();
    for (int c = 0;;) {
#pragma unroll
      for (int u = 0; u < kRows; u++) {
        const float4 f = wso[c + u * PARTS + part];
#pragma unroll
        for (int w = 0; w < 4; w++) {
          const uint32_t word = (uint32_t)q[u][w];
#pragma unroll
          for (int b = 0; b < 4; b++)
            acc[4 * w + b] = fused_term<MATH>(f, (float)((word >> (8 * b)) & 0xff), acc[4 * w + b]);
        }
      }
      c += kStep;
      if (c >= wave_cnt) break;
      request(c);
    }
    wave_lds_sync(); // slots are rewritten by the next round
  }
  if constexpr (PARTS == 2) {
#pragma unroll
    for (int c = 0; c < kCols; c++) acc[c] += __shfl_xor(acc[c], LPR, 64);
  }
  if (bag < a.segments && live && part == 0 && !alone) {
#pragma unroll
    for (int c8 = 0; c8 < kCols; c8 += 8) {
      float part8[8];
#pragma unroll
      for (int c = 0; c < 8; c++) part8[c] = acc[c8 + c];
      store_columns<8>(a, bag, (int)lane_off + c8, part8);
    }
  }
}

// A launch that does nothing (measurement: what any launch of this shape costs).
__global__ __launch_bounds__(kRowsWaves * 64) void slws_empty_kernel(float *dest) {
  if (dest == nullptr && threadIdx.x == 12345) dest[0] = 0.0f; // never taken
}

// Sum of the clamped lengths of each chunk of kChunkBags bags: one block of 1024
// threads per chunk, every length asked for in one memory trip (256 threads that
// walked the chunk length by length took sixteen dependent ones).
constexpr int kSumThreads = 1024;
__global__ __launch_bounds__(kSumThreads) void slws_chunk_sums_kernel(
    const int32_t *lengths, long long segments, int64_t *chunk_sums) {
  constexpr int kWaves = kSumThreads / 64;
  __shared__ long long s_part[kWaves];
  const long long lo = (long long)blockIdx.x * kChunkBags;
  const int n = (int)min((long long)kChunkBags, segments - lo);
  const int32_t *p = lengths + lo;
  long long sum = 0;
  if ((((uintptr_t)p) & 15) == 0) {
#pragma unroll
    for (int u = 0; u < kChunkBags / (4 * kSumThreads); u++) {
      const int i = (u * kSumThreads + (int)threadIdx.x) * 4;
      if (i + 4 <= n) {
        const int4 v = *reinterpret_cast<const int4 *>(p + i);
        sum += (long long)clamp_len(v.x) + clamp_len(v.y) + clamp_len(v.z) + clamp_len(v.w);
      } else {
        for (int k = i; k < n; k++) sum += clamp_len(p[k]);
      }
    }
  } else {
    for (int i = threadIdx.x; i < n; i += kSumThreads) sum += clamp_len(p[i]);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off, 64);
  if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    sum = 0;
#pragma unroll
    for (int w = 0; w < kWaves; w++) sum += s_part[w];
    chunk_sums[blockIdx.x] = sum;
  }
}

// Scratch for the chunk sums (lengths mode with more than kOneChunkBags bags):
// one int64 per chunk, written by slws_chunk_sums_kernel and read by the
// lookup kernel behind it on the same stream.
//
// The ordinary entry points take it from a registry keyed by (device, stream):
// launches on one stream are ordered, so they may share a buffer; launches on
// different streams never do. A buffer is allocated when the stream is made
// known to the library (mi355x_init for the device's default stream,
// mi355x_stream_create, mi355x_slws_reserve_stream), never inside a launch.
struct StreamScratch {
  int dev;
  hipStream_t stream;
  int64_t *ws;
};
static std::mutex g_ws_mutex;
static std::vector<StreamScratch> g_ws;

int slws_reserve_stream(hipStream_t st) {
  int dev = 0;
  MI355X_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(g_ws_mutex);
  for (const StreamScratch &e : g_ws)
    if (e.dev == dev && e.stream == st) return MI355X_OK;
  int64_t *ws = nullptr;
  MI355X_HIP(hipMalloc((void **)&ws, kMaxChunks * sizeof(int64_t)));
  g_ws.push_back(StreamScratch{dev, st, ws});
  return MI355X_OK;
}

int slws_release_stream(hipStream_t st) {
  int dev = 0;
  MI355X_HIP(hipGetDevice(&dev));
  int64_t *ws = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    for (size_t i = 0; i < g_ws.size(); i++)
      if (g_ws[i].dev == dev && g_ws[i].stream == st) {
        ws = g_ws[i].ws;
        g_ws.erase(g_ws.begin() + (long)i);
        break;
      }
  }
  if (ws) MI355X_HIP(hipFree(ws));
  return MI355X_OK;
}

static int stream_scratch(hipStream_t st, int64_t **ws) {
  int dev = 0;
  MI355X_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(g_ws_mutex);
  for (const StreamScratch &e : g_ws)
    if (e.dev == dev && e.stream == st) {
      *ws = e.ws;
      return MI355X_OK;
    }
  return fail(MI355X_ERR_INVALID_ARGUMENT,
              "more than %d bags on a stream without scratch for the bag offsets: "
              "use a stream from mi355x_stream_create (or the default stream after "
              "mi355x_init), or call mi355x_slws_reserve_stream(stream) once before",
              kOneChunkBags);
}

// The same scratch for callers that must not allocate: a fixed array in the
// code object, one copy per device, found once per device with
// hipGetSymbolAddress. Host code never uses the array's name as an address.
constexpr int kStaticBags = 4096 * 4096;   // 16.7M
constexpr int kStaticChunks = kStaticBags / kChunkBags;
static __device__ __align__(256) int64_t scratch[kStaticChunks];
static std::mutex g_static_mutex;
static int64_t *g_static_ptr[64] = {nullptr};

int slws_init_device() {
  int dev = 0;
  MI355X_HIP(hipGetDevice(&dev));
  MI355X_REQUIRE(dev >= 0 && dev < 64, "device index %d out of range", dev);
  std::lock_guard<std::mutex> lock(g_static_mutex);
  if (!g_static_ptr[dev]) {
    int64_t *ptr = nullptr;
    MI355X_HIP(hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch)));
    MI355X_REQUIRE(ptr, "hipGetSymbolAddress returned a NULL address");
    g_static_ptr[dev] = ptr;
  }
  return MI355X_OK;
}

static int static_scratch(int64_t **ws) {
  int dev = 0;
  MI355X_HIP(hipGetDevice(&dev));
  MI355X_REQUIRE(dev >= 0 && dev < 64, "device index %d out of range", dev);
  {
    std::lock_guard<std::mutex> lock(g_static_mutex);
    *ws = g_static_ptr[dev];
  }
  if (*ws) return MI355X_OK;
  int rc = slws_init_device();   // first call on this device
  if (rc != MI355X_OK) return rc;
  std::lock_guard<std::mutex> lock(g_static_mutex);
  *ws = g_static_ptr[dev];
  return MI355X_OK;
}

template <int LPB, int BPL>
static void launch_kind(int kind, bool acc16, dim3 grid, hipStream_t st,
                        const SlwsArgs &a) {
#define MI355X_SLWS_LAUNCH(IS4, SO16, ACC16)                                   \
  hipLaunchKernelGGL((slws_kernel<LPB, BPL, IS4, SO16, ACC16>), grid,          \
                     dim3(kSlwsThreads), 0, st, a)
  switch (kind) {
  case MI355X_FUSED_U8_F32:
    MI355X_SLWS_LAUNCH(false, false, false);
    break;
  case MI355X_FUSED_U8_F16:
    if (acc16) MI355X_SLWS_LAUNCH(false, true, true);
    else MI355X_SLWS_LAUNCH(false, true, false);
    break;
  case MI355X_FUSED_U4_F16:
    if (acc16) MI355X_SLWS_LAUNCH(true, true, true);
    else MI355X_SLWS_LAUNCH(true, true, false);
    break;
  default:
    MI355X_SLWS_LAUNCH(true, false, false);
    break;
  }
#undef MI355X_SLWS_LAUNCH
}

template <int BPL, bool OFF32>
static void launch_wave_kind(int kind, bool acc16, dim3 grid, hipStream_t st,
                             const SlwsArgs &a) {
#define MI355X_SLWS_WAVE(IS4, SO16, ACC16)                                     \
  hipLaunchKernelGGL((slws_wave_kernel<BPL, IS4, SO16, ACC16, OFF32>), grid,   \
                     dim3(kSlwsThreads), 0, st, a)
  switch (kind) {
  case MI355X_FUSED_U8_F32:
    MI355X_SLWS_WAVE(false, false, false);
    break;
  case MI355X_FUSED_U8_F16:
    if (acc16) MI355X_SLWS_WAVE(false, true, true);
    else MI355X_SLWS_WAVE(false, true, false);
    break;
  case MI355X_FUSED_U4_F16:
    if (acc16) MI355X_SLWS_WAVE(true, true, true);
    else MI355X_SLWS_WAVE(true, true, false);
    break;
  default:
    MI355X_SLWS_WAVE(true, false, false);
    break;
  }
#undef MI355X_SLWS_WAVE
}

template <int LPR, bool OFF32, int MATH, int WAVES>
static void launch_rows_kind(int kind, dim3 grid, hipStream_t st, const SlwsArgs &a) {
#define MI355X_SLWS_ROWS(IS4, SO16)                                            \
  hipLaunchKernelGGL((slws_rows_kernel<IS4, SO16, LPR, OFF32, MATH, WAVES>), grid, \
                     dim3(WAVES * 64), 0, st, a)
  switch (kind) {
  case MI355X_FUSED_U8_F32:
    MI355X_SLWS_ROWS(false, false);
    break;
  case MI355X_FUSED_U8_F16:
    MI355X_SLWS_ROWS(false, true);
    break;
  case MI355X_FUSED_U4_F16:
    MI355X_SLWS_ROWS(true, true);
    break;
  default:
    MI355X_SLWS_ROWS(true, false);
    break;
  }
#undef MI355X_SLWS_ROWS
}

// (32 lanes to a row: rounds of 64 lookups; 64 lanes, a load instruction per row: of 32)
template <int LPR>
static void launch_ranges_kind(int kind, dim3 grid, hipStream_t st, const SlwsArgs &a, int per_block) {
#define MI355X_SLWS_RANGES(IS4, SO16)                                          \
  hipLaunchKernelGGL((slws_ranges_kernel<IS4, SO16, LPR, true, kMathElement, kRangesWaves,       \
                                         2048 / LPR>),                         \
                     grid, dim3(kRangesWaves * 64), 0, st, a, per_block)
  switch (kind) {
  case MI355X_FUSED_U8_F32:
    MI355X_SLWS_RANGES(false, false);
    break;
  case MI355X_FUSED_U8_F16:
    MI355X_SLWS_RANGES(false, true);
    break;
  case MI355X_FUSED_U4_F16:
    MI355X_SLWS_RANGES(true, true);
    break;
  default:
    MI355X_SLWS_RANGES(true, false);
    break;
  }
#undef MI355X_SLWS_RANGES
}

template <int LPR, bool OFF32, int MATH, int BPL = 4>
static void launch_groups_kind(int kind, dim3 grid, hipStream_t st, const SlwsArgs &a) {
#define MI355X_SLWS_GROUPS(IS4, SO16)                                          \
  hipLaunchKernelGGL((slws_groups_kernel<IS4, SO16, LPR, OFF32, MATH, BPL>), grid, \
                     dim3(kSlwsThreads), 0, st, a)
  switch (kind) {
  case MI355X_FUSED_U8_F32:
    MI355X_SLWS_GROUPS(false, false);
    break;
  case MI355X_FUSED_U8_F16:
    MI355X_SLWS_GROUPS(false, true);
    break;
  case MI355X_FUSED_U4_F16:
    MI355X_SLWS_GROUPS(true, true);
    break;
  default:
    MI355X_SLWS_GROUPS(true, false);
    break;
  }
#undef MI355X_SLWS_GROUPS
}

template <int LPR, int PARTS, int MATH>
static void launch_wide(bool so16, dim3 grid, hipStream_t st, const SlwsArgs &a) {
  if (so16)
    hipLaunchKernelGGL((slws_wide_kernel<true, LPR, PARTS, MATH>), grid, dim3(kSlwsThreads), 0, st, a);
  else
    hipLaunchKernelGGL((slws_wide_kernel<false, LPR, PARTS, MATH>), grid, dim3(kSlwsThreads), 0, st, a);
}

// Arithmetic of the launches that do not name one (process-wide default).
static std::atomic<int> g_fused_math{kMathElement};
// Arithmetic named by the call being issued on this thread (OptsScope); -1: none.
thread_local int g_slws_math = -1;

// Several tables in one launch and/or the int8 output transform.
struct SlwsExtra {
  const float *sep_scales = nullptr, *sep_offsets = nullptr; // rowwise tables
  const mi355x_sls_table *tables = nullptr; // device array
  size_t n_tables = 1;
  int out_q8 = 0;
  float q_scale = 1.0f;
  int32_t q_offset = 0;
  size_t q_stride = 0;
  bool static_scratch = false; // chunk sums in the code object's fixed array
  int math = -1;               // kMath*; -1 = the process-wide default
  int probe = kProbeOff;       // measurement cut point (mi355x_frwq_slws_probe)
};

static int slws_dispatch(void *dest, int out_is_f16, const uint8_t *data,
                         size_t data_rows, int kind, const void *weights,
                         int weights_are_f16, const void *indices,
                         int idx_is_64, size_t num_indices,
                         const int32_t *lengths, const int32_t *offsets,
                         int has_end_offset, size_t out_rows,
                         size_t in_line_size, size_t out_line_size,
                         int fp16_accum, void *stream,
                         const SlwsExtra &x = SlwsExtra()) {
  if (out_rows == 0 || x.n_tables == 0) return MI355X_OK;
  MI355X_REQUIRE(kind >= 0 && kind <= 3, "unknown fused kind %d", kind);
  MI355X_REQUIRE(x.tables || (dest && (lengths || offsets)), "NULL tensor");
  MI355X_REQUIRE(x.n_tables <= 65535, "more than 65535 tables");
  const bool is4 = kind == MI355X_FUSED_U4_F16 || kind == MI355X_FUSED_U4_F32;
  const bool so16 = kind == MI355X_FUSED_U8_F16 || kind == MI355X_FUSED_U4_F16;
  const size_t so_bytes = x.sep_scales ? 0 : (so16 ? 4 : 8);
  // in_line_size is the distance between rows: the fused row's own size, or
  // more when the table has been laid out with padded rows
  MI355X_REQUIRE(out_line_size > 0 && (!is4 || out_line_size % 2 == 0),
                 "out_line_size %zu is not a row of this kind", out_line_size);
  const size_t cols = out_line_size;
  const size_t data_bytes = is4 ? cols / 2 : cols;
  MI355X_REQUIRE(in_line_size >= data_bytes + so_bytes,
                 "in_line_size %zu does not hold %zu columns of the fused row",
                 in_line_size, cols);
  MI355X_REQUIRE(in_line_size < (1u << 20) && data_rows < (1ull << 31) &&
                     out_rows < (1ull << 40),
                 "table or batch too large");
  MI355X_REQUIRE(x.tables || num_indices == 0 || (indices && data),
                 "NULL indices or data with num_indices > 0");
  MI355X_REQUIRE(!x.tables || out_rows <= (size_t)kTableBags,
                 "a multi-table launch takes at most %d bags per table", kTableBags);
  MI355X_REQUIRE(!x.out_q8 || x.q_stride >= cols, "output rows overlap");
  hipStream_t st = as_stream(stream);

  SlwsArgs a;
  a.dest = dest;
  a.data = data;
  a.weights = weights;
  a.indices = indices;
  a.lengths = lengths;
  a.offsets = offsets;
  a.chunk_sums = nullptr;
  a.data_rows = (int64_t)data_rows;
  a.num_indices = (int64_t)num_indices;
  a.segments = (int64_t)out_rows;
  a.offsets_have_end = has_end_offset;
  a.in_line = (int32_t)in_line_size;
  a.data_bytes = (int32_t)data_bytes;
  a.out_cols = (int32_t)cols;
  a.out16 = out_is_f16;
  a.w16 = weights_are_f16;
  a.idx64 = idx_is_64;
  a.sep_scales = x.sep_scales;
  a.sep_offsets = x.sep_offsets;
  a.tables = x.tables;
  a.out_q8 = x.out_q8;
  a.q_scale = x.q_scale;
  a.q_offset = (float)x.q_offset;
  a.q_stride = (int64_t)x.q_stride;
  a.long_bag = 0;

  const bool acc16 = out_is_f16 && fp16_accum && so16;
  const bool even = (in_line_size % 2 == 0) && (((uintptr_t)data) % 2 == 0);
  int lpb = 64;
  if (even && data_bytes <= 32) lpb = 16;
  else if (even && data_bytes <= 64) lpb = 32;
  const size_t groups = kSlwsThreads / lpb;
  const size_t blocks = (out_rows + groups - 1) / groups;
  MI355X_REQUIRE(blocks < 0x7fffffffu, "too many bags");
  dim3 grid((unsigned)blocks, (unsigned)x.n_tables);
  const bool off32 = (unsigned long long)data_rows * in_line_size <= 0xffffffffull;
  // rows read a word per lane: a multiple of 4 data bytes, 4-byte aligned rows,
  // fp32 accumulation. A multi-table launch cannot check the alignment of each
  // table here; its tables must be 4-byte aligned.
  const int math = x.math >= 0     ? x.math
                   : g_slws_math >= 0 ? g_slws_math
                                      : g_fused_math.load(std::memory_order_relaxed);
  MI355X_REQUIRE(math >= kMathStrict && math <= kMathRegrouped,
                 "unknown SparseLengths arithmetic %d", math);
  const bool words = !acc16 && in_line_size % 4 == 0 && (((uintptr_t)data) % 4 == 0) &&
                     data_bytes % 4 == 0;
  // the fused arithmetic covers rows of 32 to 256 data bytes; narrower rows keep
  // the CPU loop's separately rounded operations whatever is asked for
  const bool rows_ok = words && math != kMathStrict && data_bytes >= 32 && data_bytes <= 256;
  // enough bags to fill the chip with several per wavefront
  const bool many = out_rows * x.n_tables > kShortRowsWaveBags;
  const size_t mean = num_indices / std::max<size_t>(out_rows, 1);
  // (the kernels for many bags; why the lines lie there: where they are launched)
  const bool wide_ok = !is4 && !acc16 && off32 && !x.tables && out_rows > kWideBags && data_bytes > 32 &&
      data_bytes <= 256 &&
      (words ? rows_ok && math == kMathElement && data_bytes > 64 && data_bytes <= 128 &&
                   mean <= kWideLen && mean * data_bytes <= kWideBytes
             : mean <= kWideAnyLen || (out_rows >= kWideAnyBags && data_bytes > 64));
  // More bags than fit a wavefront each at once: the wavefronts take them in turns. Not long
  // ones, whose rows alone fill the chip, where fewer wavefronts are resident that way.
  const bool long_bags = is4 ? mean >= kRangesLen4
                             : data_bytes <= 128 && mean >= kRangesLen128 && out_rows > kRangesBags128;
  const size_t beyond =
      data_bytes > 128 && mean >= kRangesLenWide ? (is4 ? kRangesBags : kRangesBagsEarly)
      : is4 || (data_bytes <= 128 && kind != MI355X_FUSED_U8_F16) ? kRangesBagsLate
                                                                  : kRangesBags;
  const bool ranges = !wide_ok && x.probe == kProbeOff && rows_ok && math == kMathElement && off32 &&
      !x.tables && data_bytes > 64 && out_rows > beyond && !long_bags &&
      (data_bytes > 128 || kind == MI355X_FUSED_U8_F16 || out_rows > kRangesBags128 ||
       out_rows <= kRangesBags64);

  if (!offsets) {
    const size_t chunks = (out_rows + kChunkBags - 1) / kChunkBags;
    if (out_rows > (size_t)kOneChunkBags) {
      int64_t *ws = nullptr;
      int rc;
      if (x.static_scratch) {
        MI355X_REQUIRE(out_rows <= (size_t)kStaticBags,
                       "%zu bags: the entry point that allocates nothing takes at "
                       "most %d", out_rows, kStaticBags);
        rc = static_scratch(&ws);
      } else {
        MI355X_REQUIRE(chunks <= (size_t)kMaxChunks, "more than %d bags",
                       kMaxChunks * kChunkBags);
        rc = stream_scratch(st, &ws);
      }
      if (rc != MI355X_OK) return rc;
      // (what is asked of a stream goes by the bags alone; the kernel that sums up to
      // kRangesOneBags lengths itself leaves its scratch alone)
      if (!ranges || out_rows > (size_t)kRangesOneBags) {
        hipLaunchKernelGGL(slws_chunk_sums_kernel, dim3((unsigned)chunks),
                           dim3(kSumThreads), 0, st, lengths, (long long)out_rows, ws);
        rc = check_launch("slws_chunk_sums");
        if (rc != MI355X_OK) return rc;
        a.chunk_sums = ws;
      }
    }
  }

  if (x.probe != kProbeOff) {
    MI355X_REQUIRE(rows_ok && kind == MI355X_FUSED_U8_F32 && data_bytes == 128 && off32 &&
                       !x.tables && !x.out_q8 && math == kMathElement,
                   "the probe covers uint8 rows of 128 columns with fp32 scale and offset");
    const size_t pw = (size_t)rows_waves(out_rows);
    const size_t rblocks = (out_rows + pw - 1) / pw;
    MI355X_REQUIRE(rblocks < 0x7fffffffu, "too many bags");
    dim3 rgrid((unsigned)rblocks);
#define MI355X_PROBE_CASE(P)                                                   \
  case P:                                                                      \
    if (pw == (size_t)kRowsWavesFew)                                           \
      hipLaunchKernelGGL(                                                      \
          (slws_rows_kernel<false, false, 32, true, kMathElement, kRowsWavesFew, P>), rgrid, \
          dim3(kRowsWavesFew * 64), 0, st, a);                                 \
    else if (pw == (size_t)kRowsWaves)                                         \
      hipLaunchKernelGGL(                                                      \
          (slws_rows_kernel<false, false, 32, true, kMathElement, kRowsWaves, P>), rgrid, \
          dim3(kRowsWaves * 64), 0, st, a);                                    \
    else                                                                       \
      hipLaunchKernelGGL(                                                      \
          (slws_rows_kernel<false, false, 32, true, kMathElement, kRowsWavesMany, P>), rgrid, \
          dim3(kRowsWavesMany * 64), 0, st, a);                                \
    break;
    switch (x.probe) {
      MI355X_PROBE_CASE(kProbeSpan)
      MI355X_PROBE_CASE(kProbeIndex)
      MI355X_PROBE_CASE(kProbeScaleOffset)
      MI355X_PROBE_CASE(kProbeRows)
    default:
      return fail(MI355X_ERR_INVALID_ARGUMENT, "unknown probe stage %d", x.probe);
    }
#undef MI355X_PROBE_CASE
    return check_launch("frwq_slws_probe");
  }
  // Many short bags of eight-bit rows, sixteen bytes of a row to a lane and several bags side
  // by side in a wavefront: a bag per wavefront at a time is a first pass and a sum across
  // lanes for a few rows, and rows that start at any byte are read a byte or two to a lane
  // there. us, the kernels below / this one, Poisson lengths and indices all over a table of a
  // million rows, bags x mean: 100 columns 13 000 x 3 8.6 / 7.5, 20 000 x 4 11.8 / 11.2, 40 000 x
  // 4 18.5 / 17.0, 60 000 x 9 27.5 / 26.8, 128 columns 60 000 x 4 25.3 / 23.8; 101 columns, at any
  // byte, 13 000 x 3 18.8 / 12.1, 30 000 x 12 48.5 / 36.5. The lines, likewise: 128 columns 16 300
  // x 8 10.7 / 10.6, 30 000 x 6 15.0 / 16.4, 40 000 x 6 19.0 / 19.2, 100 columns 20 000 x 8 12.8 /
  // 12.7, 30 000 x 8 15.5 / 16.6, 68 columns 30 000 x 12 16.4 / 17.7; rows of more than 128 bytes, 200 columns
  // 30 000 x 4 16.2 / 19.6; any byte, 33 columns 30 000 x 12 34.2 / 28.1, x 30 44.3 / 50.1,
  // 101 columns x 30 68.9 / 65.0. Four-bit rows, twice the registers here, won 7 % at best
  // and lost 30 % with uneven bags.
  if (wide_ok) {
    const int lpr = data_bytes <= 64 ? 4 : data_bytes <= 128 ? 8 : 16;
    const size_t per_block = (size_t)(kSlwsThreads / lpr) / (words ? 2 : 1);
    const size_t wblocks = (out_rows + per_block - 1) / per_block;
    MI355X_REQUIRE(wblocks < 0x7fffffffu, "too many bags");
    const dim3 wgrid((unsigned)wblocks);
    a.long_bag = (int32_t)std::min<size_t>(std::max<size_t>(kLongBag, kLongBagMeans * mean), 1 << 30);
    if (words) {
      launch_wide<8, 2, kMathElement>(so16, wgrid, st, a);
    } else {
      if (lpr == 4) launch_wide<4, 1, kMathStrict>(so16, wgrid, st, a);
      else if (lpr == 8) launch_wide<8, 1, kMathStrict>(so16, wgrid, st, a);
      else launch_wide<16, 1, kMathStrict>(so16, wgrid, st, a);
    }
    return check_launch("frwq_slws");
  }
  if (words && data_bytes <= 64 && (!rows_ok || many)) {
    // short rows, several bags per wavefront: in bag order per lane, which the
    // strict arithmetic needs too
    const bool bytewise = data_bytes < 32 && !(out_rows * x.n_tables > kByteLaneBags);
    const int lpr = (data_bytes <= 16 ? 4 : data_bytes <= 32 ? 8 : 16) * (bytewise ? 4 : 1);
    const size_t per_block = kSlwsThreads / lpr;
    const size_t gblocks = (out_rows + per_block - 1) / per_block;
    MI355X_REQUIRE(gblocks < 0x7fffffffu, "too many bags");
    dim3 ggrid((unsigned)gblocks, (unsigned)x.n_tables);
#define MI355X_GROUPS_MATH(LPR, MATH)                                          \
  if (off32) launch_groups_kind<LPR, true, MATH>(kind, ggrid, st, a);          \
  else launch_groups_kind<LPR, false, MATH>(kind, ggrid, st, a);
#define MI355X_GROUPS_CASE(LPR)                                                \
  if (!rows_ok) {                                                              \
    MI355X_GROUPS_MATH(LPR, kMathStrict)                                       \
  } else if (math == kMathElement) {                                           \
    MI355X_GROUPS_MATH(LPR, kMathElement)                                      \
  } else {                                                                     \
    MI355X_GROUPS_MATH(LPR, kMathRegrouped)                                    \
  }
    if (bytewise) {
#define MI355X_GROUPS_BYTES(LPR)                                               \
  if (off32) launch_groups_kind<LPR, true, kMathStrict, 1>(kind, ggrid, st, a); \
  else launch_groups_kind<LPR, false, kMathStrict, 1>(kind, ggrid, st, a);
      if (lpr == 16) {
        MI355X_GROUPS_BYTES(16)
      } else {
        MI355X_GROUPS_BYTES(32)
      }
#undef MI355X_GROUPS_BYTES
    } else if (lpr == 4) {
      MI355X_GROUPS_MATH(4, kMathStrict)
    } else if (lpr == 8) {
      MI355X_GROUPS_CASE(8)
    } else {
      MI355X_GROUPS_CASE(16)
    }
#undef MI355X_GROUPS_CASE
#undef MI355X_GROUPS_MATH
    return check_launch("frwq_slws");
  }
  if (ranges) {
    // as many blocks as are resident at once, or a multiple of that where one takes the 64
    // bags of its table; whole turns of its wavefronts, of four-bit rows fours of bags
    const size_t resident = is4 && (data_bytes > 128 || !so16) ? kRangesBlocks4 : kRangesBlocks;
    const size_t whole = is4 ? 4 : kRangesWaves;
    const size_t rounds = (out_rows + 64 * resident - 1) / (64 * resident);
    const size_t share = (out_rows + resident * rounds - 1) / (resident * rounds);
    const int per_block = (int)((share + whole - 1) / whole * whole);
    const size_t rblocks = (out_rows + per_block - 1) / per_block;
    MI355X_REQUIRE(rblocks < 0x7fffffffu, "too many bags");
    if (data_bytes <= 128) launch_ranges_kind<32>(kind, dim3((unsigned)rblocks), st, a, per_block);
    else launch_ranges_kind<64>(kind, dim3((unsigned)rblocks), st, a, per_block);
    return check_launch("frwq_slws");
  }
  if (rows_ok) {
    // a bag per wavefront, as many lanes per row as the row has words (rounded
    // up to a power of two)
    const size_t rw = (size_t)rows_waves(out_rows * x.n_tables);
    const size_t rblocks = (out_rows + rw - 1) / rw;
    MI355X_REQUIRE(rblocks < 0x7fffffffu, "too many bags");
    dim3 rgrid((unsigned)rblocks, (unsigned)x.n_tables);
#define MI355X_ROWS_OFF(LPR, MATH, WAVES)                                      \
  if (off32) launch_rows_kind<LPR, true, MATH, WAVES>(kind, rgrid, st, a);     \
  else launch_rows_kind<LPR, false, MATH, WAVES>(kind, rgrid, st, a);
#define MI355X_ROWS_WAVES(LPR, WAVES)                                          \
  if (math == kMathElement) {                                                  \
    MI355X_ROWS_OFF(LPR, kMathElement, WAVES)                                  \
  } else {                                                                     \
    MI355X_ROWS_OFF(LPR, kMathRegrouped, WAVES)                                \
  }
// short rows: not with more than kShortRowsWaveBags bags
#define MI355X_ROWS_FEW(LPR)                                                   \
  if (rw == (size_t)kRowsWavesFew) {                                           \
    MI355X_ROWS_WAVES(LPR, kRowsWavesFew)                                      \
  } else {                                                                     \
    MI355X_ROWS_WAVES(LPR, kRowsWaves)                                         \
  }
#define MI355X_ROWS_LPR(LPR)                                                   \
  if (rw == (size_t)kRowsWavesFew) {                                           \
    MI355X_ROWS_WAVES(LPR, kRowsWavesFew)                                      \
  } else if (rw == (size_t)kRowsWaves) {                                       \
    MI355X_ROWS_WAVES(LPR, kRowsWaves)                                         \
  } else {                                                                     \
    MI355X_ROWS_WAVES(LPR, kRowsWavesMany)                                     \
  }
    if (data_bytes <= 32) {
      MI355X_ROWS_FEW(8)
    } else if (data_bytes <= 64) {
      MI355X_ROWS_FEW(16)
    } else if (data_bytes <= 128) {
      MI355X_ROWS_LPR(32)
    } else {
      MI355X_ROWS_LPR(64)
    }
#undef MI355X_ROWS_LPR
#undef MI355X_ROWS_FEW
#undef MI355X_ROWS_WAVES
#undef MI355X_ROWS_OFF
    return check_launch("frwq_slws");
  }
  if (lpb == 16) launch_kind<16, 2>(kind, acc16, grid, st, a);
  else if (lpb == 32) launch_kind<32, 2>(kind, acc16, grid, st, a);
  else if (!even && off32) launch_wave_kind<1, true>(kind, acc16, grid, st, a);
  else if (!even) launch_wave_kind<1, false>(kind, acc16, grid, st, a);
  else if (off32) launch_wave_kind<2, true>(kind, acc16, grid, st, a);
  else launch_wave_kind<2, false>(kind, acc16, grid, st, a);
  return check_launch("frwq_slws");
}

} // namespace mi355x

using namespace mi355x;

extern "C" {

int mi355x_slws_set_fused_math(int on) {  // on: MI355X_SLWS_MATH_*
  MI355X_REQUIRE(on >= kMathStrict && on <= kMathRegrouped,
                 "unknown SparseLengths arithmetic %d", on);
  g_fused_math.store(on, std::memory_order_relaxed);
  return MI355X_OK;
}

int mi355x_frwq_slws_probe(int stage, float *dest, const uint8_t *data, size_t data_rows,
                           const float *weights, const int64_t *indices,
                           size_t num_indices, const int32_t *lengths, size_t segments,
                           size_t in_line_size, void *stream) {
  MI355X_REQUIRE(segments == 0 || lengths, "lengths is NULL");
  if (stage == 0) {
    // a launch of the same shape that does nothing
    if (segments == 0) return MI355X_OK;
    const size_t w = (size_t)rows_waves(segments);
    hipLaunchKernelGGL(slws_empty_kernel, dim3((unsigned)((segments + w - 1) / w)),
                       dim3((unsigned)w * 64), 0, as_stream(stream), dest);
    return check_launch("slws_empty");
  }
  SlwsExtra x;
  x.math = kMathElement;
  x.probe = stage;
  return slws_dispatch(dest, 0, data, data_rows, MI355X_FUSED_U8_F32, weights, 0, indices, 1,
                       num_indices, lengths, nullptr, 0, segments, in_line_size, 128, 0,
                       stream, x);
}

static int mi355x_frwq_sls_multi_impl(const mi355x_sls_table *tables, size_t n_tables,
                          size_t max_data_rows, int kind, int idx_is_64,
                          size_t segments, size_t in_line_size,
                          size_t out_line_size, int out_kind, float out_scale,
                          int32_t out_offset, size_t dest_row_stride,
                          int fp16_accum, void *stream) {
  if (n_tables == 0 || segments == 0) return MI355X_OK;
  MI355X_REQUIRE(tables, "tables is NULL");
  MI355X_REQUIRE(out_kind >= 0 && out_kind <= 3, "unknown output kind %d", out_kind);
  SlwsExtra x;
  x.tables = tables;
  x.n_tables = n_tables;
  x.out_q8 = out_kind >= 2;
  x.q_scale = out_scale;
  x.q_offset = out_offset;
  x.q_stride = dest_row_stride;
  const int out16 = out_kind == MI355X_SLS_OUT_F16 || out_kind == MI355X_SLS_OUT_I8_VIA_F16;
  return slws_dispatch(nullptr, out16, nullptr, max_data_rows, kind, nullptr, 0, nullptr,
                       idx_is_64, 0, nullptr, nullptr, 0, segments, in_line_size,
                       out_line_size, fp16_accum, stream, x);
}

int mi355x_frwq_sls_multi(const mi355x_sls_table *tables, size_t n_tables,
                          size_t max_data_rows, int kind, int idx_is_64,
                          size_t segments, size_t in_line_size,
                          size_t out_line_size, int out_kind, float out_scale,
                          int32_t out_offset, size_t dest_row_stride,
                          int fp16_accum, void *stream) {
  return mi355x_frwq_sls_multi_impl(tables, n_tables, max_data_rows, kind, idx_is_64, segments, in_line_size, out_line_size, out_kind, out_scale, out_offset, dest_row_stride, fp16_accum, stream);
}

int mi355x_frwq_sls_multi_opts(const mi355x_sls_table *tables, size_t n_tables,
                          size_t max_data_rows, int kind, int idx_is_64,
                          size_t segments, size_t in_line_size,
                          size_t out_line_size, int out_kind, float out_scale,
                          int32_t out_offset, size_t dest_row_stride,
                          int fp16_accum, void *stream,
    const mi355x_launch_opts *opts) {
  OptsScope scope(opts);
  if (scope.rc != MI355X_OK) return scope.rc;
  return mi355x_frwq_sls_multi_impl(tables, n_tables, max_data_rows, kind, idx_is_64, segments, in_line_size, out_line_size, out_kind, out_scale, out_offset, dest_row_stride, fp16_accum, stream);
}

static int mi355x_rwq_slws_impl(float *dest, const uint8_t *data, size_t data_rows,
                    const float *scales, const float *offsets, const float *weights,
                    const void *indices, int idx_is_64, size_t num_indices,
                    const int32_t *lengths, size_t segments, size_t line_size,
                    void *stream) {
  MI355X_REQUIRE(segments == 0 || lengths, "lengths is NULL");
  MI355X_REQUIRE(segments == 0 || (scales && offsets), "NULL scales or offsets");
  SlwsExtra x;
  x.sep_scales = scales;
  x.sep_offsets = offsets;
  return slws_dispatch(dest, 0, data, data_rows, MI355X_FUSED_U8_F32, weights, 0, indices,
                       idx_is_64, num_indices, lengths, nullptr, 0, segments, line_size,
                       line_size, 0, stream, x);
}

int mi355x_rwq_slws(float *dest, const uint8_t *data, size_t data_rows,
                    const float *scales, const float *offsets, const float *weights,
                    const void *indices, int idx_is_64, size_t num_indices,
                    const int32_t *lengths, size_t segments, size_t line_size,
                    void *stream) {
  return mi355x_rwq_slws_impl(dest, data, data_rows, scales, offsets, weights, indices, idx_is_64, num_indices, lengths, segments, line_size, stream);
}

int mi355x_rwq_slws_opts(float *dest, const uint8_t *data, size_t data_rows,
                    const float *scales, const float *offsets, const float *weights,
                    const void *indices, int idx_is_64, size_t num_indices,
                    const int32_t *lengths, size_t segments, size_t line_size,
                    void *stream,
    const mi355x_launch_opts *opts) {
  OptsScope scope(opts);
  if (scope.rc != MI355X_OK) return scope.rc;
  return mi355x_rwq_slws_impl(dest, data, data_rows, scales, offsets, weights, indices, idx_is_64, num_indices, lengths, segments, line_size, stream);
}

static int mi355x_frwq_slws_impl(void *dest, int out_is_f16, const uint8_t *data,
                     size_t data_rows, int kind, const void *weights,
                     int weights_are_f16, const void *indices, int idx_is_64,
                     size_t num_indices, const int32_t *lengths,
                     size_t segments, size_t in_line_size,
                     size_t out_line_size, int fp16_accum, void *stream) {
  MI355X_REQUIRE(segments == 0 || lengths, "lengths is NULL");
  return slws_dispatch(dest, out_is_f16, data, data_rows, kind, weights,
                       weights_are_f16, indices, idx_is_64, num_indices,
                       lengths, nullptr, 0, segments, in_line_size,
                       out_line_size, fp16_accum, stream);
}

int mi355x_frwq_slws(void *dest, int out_is_f16, const uint8_t *data,
                     size_t data_rows, int kind, const void *weights,
                     int weights_are_f16, const void *indices, int idx_is_64,
                     size_t num_indices, const int32_t *lengths,
                     size_t segments, size_t in_line_size,
                     size_t out_line_size, int fp16_accum, void *stream) {
  return mi355x_frwq_slws_impl(dest, out_is_f16, data, data_rows, kind, weights, weights_are_f16, indices, idx_is_64, num_indices, lengths, segments, in_line_size, out_line_size, fp16_accum, stream);
}

int mi355x_frwq_slws_opts(void *dest, int out_is_f16, const uint8_t *data,
                     size_t data_rows, int kind, const void *weights,
                     int weights_are_f16, const void *indices, int idx_is_64,
                     size_t num_indices, const int32_t *lengths,
                     size_t segments, size_t in_line_size,
                     size_t out_line_size, int fp16_accum, void *stream,
    const mi355x_launch_opts *opts) {
  OptsScope scope(opts);
  if (scope.rc != MI355X_OK) return scope.rc;
  return mi355x_frwq_slws_impl(dest, out_is_f16, data, data_rows, kind, weights, weights_are_f16, indices, idx_is_64, num_indices, lengths, segments, in_line_size, out_line_size, fp16_accum, stream);
}

static int mi355x_frwq_slws_noalloc_impl(void *dest, int out_is_f16, const uint8_t *data,
                             size_t data_rows, int kind, const void *weights,
                             int weights_are_f16, const void *indices, int idx_is_64,
                             size_t num_indices, const int32_t *lengths,
                             size_t segments, size_t in_line_size,
                             size_t out_line_size, int fp16_accum, void *stream) {
  MI355X_REQUIRE(segments == 0 || lengths, "lengths is NULL");
  MI355X_REQUIRE(segments <= (size_t)kStaticBags,
                 "%zu bags: mi355x_frwq_slws_noalloc takes at most %d", segments, kStaticBags);
  SlwsExtra x;
  x.static_scratch = true;
  return slws_dispatch(dest, out_is_f16, data, data_rows, kind, weights,
                       weights_are_f16, indices, idx_is_64, num_indices,
                       lengths, nullptr, 0, segments, in_line_size,
                       out_line_size, fp16_accum, stream, x);
}

int mi355x_frwq_slws_noalloc(void *dest, int out_is_f16, const uint8_t *data,
                             size_t data_rows, int kind, const void *weights,
                             int weights_are_f16, const void *indices, int idx_is_64,
                             size_t num_indices, const int32_t *lengths,
                             size_t segments, size_t in_line_size,
                             size_t out_line_size, int fp16_accum, void *stream) {
  return mi355x_frwq_slws_noalloc_impl(dest, out_is_f16, data, data_rows, kind, weights, weights_are_f16, indices, idx_is_64, num_indices, lengths, segments, in_line_size, out_line_size, fp16_accum, stream);
}

int mi355x_frwq_slws_noalloc_opts(void *dest, int out_is_f16, const uint8_t *data,
                             size_t data_rows, int kind, const void *weights,
                             int weights_are_f16, const void *indices, int idx_is_64,
                             size_t num_indices, const int32_t *lengths,
                             size_t segments, size_t in_line_size,
                             size_t out_line_size, int fp16_accum, void *stream,
    const mi355x_launch_opts *opts) {
  OptsScope scope(opts);
  if (scope.rc != MI355X_OK) return scope.rc;
  return mi355x_frwq_slws_noalloc_impl(dest, out_is_f16, data, data_rows, kind, weights, weights_are_f16, indices, idx_is_64, num_indices, lengths, segments, in_line_size, out_line_size, fp16_accum, stream);
}

static int mi355x_frwq_slws_offsets_impl(void *dest, int out_is_f16, const uint8_t *data,
                             size_t data_rows, int kind, const void *weights,
                             int weights_are_f16, const void *indices, int idx_is_64,
                             size_t num_indices, const int32_t *bag_offsets,
                             size_t segments, size_t in_line_size,
                             size_t out_line_size, int fp16_accum, void *stream) {
  MI355X_REQUIRE(segments == 0 || bag_offsets, "bag_offsets is NULL");
  // segments + 1 offsets: every bag reads its two ends, no prefix sum, no
  // scratch and no second launch whatever the number of bags
  return slws_dispatch(dest, out_is_f16, data, data_rows, kind, weights,
                       weights_are_f16, indices, idx_is_64, num_indices, nullptr,
                       bag_offsets, 1, segments, in_line_size, out_line_size,
                       fp16_accum, stream);
}

int mi355x_frwq_slws_offsets(void *dest, int out_is_f16, const uint8_t *data,
                             size_t data_rows, int kind, const void *weights,
                             int weights_are_f16, const void *indices, int idx_is_64,
                             size_t num_indices, const int32_t *bag_offsets,
                             size_t segments, size_t in_line_size,
                             size_t out_line_size, int fp16_accum, void *stream) {
  return mi355x_frwq_slws_offsets_impl(dest, out_is_f16, data, data_rows, kind, weights, weights_are_f16, indices, idx_is_64, num_indices, bag_offsets, segments, in_line_size, out_line_size, fp16_accum, stream);
}

int mi355x_frwq_slws_offsets_opts(void *dest, int out_is_f16, const uint8_t *data,
                             size_t data_rows, int kind, const void *weights,
                             int weights_are_f16, const void *indices, int idx_is_64,
                             size_t num_indices, const int32_t *bag_offsets,
                             size_t segments, size_t in_line_size,
                             size_t out_line_size, int fp16_accum, void *stream,
    const mi355x_launch_opts *opts) {
  OptsScope scope(opts);
  if (scope.rc != MI355X_OK) return scope.rc;
  return mi355x_frwq_slws_offsets_impl(dest, out_is_f16, data, data_rows, kind, weights, weights_are_f16, indices, idx_is_64, num_indices, bag_offsets, segments, in_line_size, out_line_size, fp16_accum, stream);
}

int mi355x_slws_bag_offsets_host(const int32_t *lengths, size_t segments,
                                 int32_t *bag_offsets) {
  MI355X_REQUIRE(bag_offsets && (segments == 0 || lengths), "NULL vector");
  uint64_t sum = 0;
  bag_offsets[0] = 0;
  for (size_t i = 0; i < segments; i++) {
    sum += lengths[i] > 0 ? (uint64_t)lengths[i] : 0u;   // as the kernels clamp
    MI355X_REQUIRE(sum <= 0x7fffffffull,
                   "the lengths sum past 2^31 - 1 at bag %zu: use the lengths entry point", i);
    bag_offsets[i + 1] = (int32_t)sum;
  }
  return MI355X_OK;
}

int mi355x_slws_reserve_stream(void *stream) {
  return slws_reserve_stream(as_stream(stream));
}

static int mi355x_embedding_bag_rowwise_offsets_impl(
    void *dest, int out_is_f16, const uint8_t *data, size_t data_rows,
    int kind, const void *weights, int weights_are_f16, const int32_t *indices,
    size_t num_indices, const int32_t *offsets, size_t segments,
    int has_end_offset, size_t in_line_size, size_t out_line_size,
    int fp16_accum, void *stream) {
  MI355X_REQUIRE(segments == 0 || offsets, "offsets is NULL");
  if (has_end_offset) {
    MI355X_REQUIRE(segments >= 1, "has_end_offset needs at least one offset");
    segments -= 1;
  }
  return slws_dispatch(dest, out_is_f16, data, data_rows, kind, weights,
                       weights_are_f16, indices, 0, num_indices, nullptr,
                       offsets, has_end_offset, segments, in_line_size,
                       out_line_size, fp16_accum, stream);
}

int mi355x_embedding_bag_rowwise_offsets(
    void *dest, int out_is_f16, const uint8_t *data, size_t data_rows,
    int kind, const void *weights, int weights_are_f16, const int32_t *indices,
    size_t num_indices, const int32_t *offsets, size_t segments,
    int has_end_offset, size_t in_line_size, size_t out_line_size,
    int fp16_accum, void *stream) {
  return mi355x_embedding_bag_rowwise_offsets_impl(dest, out_is_f16, data, data_rows, kind, weights, weights_are_f16, indices, num_indices, offsets, segments, has_end_offset, in_line_size, out_line_size, fp16_accum, stream);
}

int mi355x_embedding_bag_rowwise_offsets_opts(
    void *dest, int out_is_f16, const uint8_t *data, size_t data_rows,
    int kind, const void *weights, int weights_are_f16, const int32_t *indices,
    size_t num_indices, const int32_t *offsets, size_t segments,
    int has_end_offset, size_t in_line_size, size_t out_line_size,
    int fp16_accum, void *stream,
    const mi355x_launch_opts *opts) {
  OptsScope scope(opts);
  if (scope.rc != MI355X_OK) return scope.rc;
  return mi355x_embedding_bag_rowwise_offsets_impl(dest, out_is_f16, data, data_rows, kind, weights, weights_are_f16, indices, num_indices, offsets, segments, has_end_offset, in_line_size, out_line_size, fp16_accum, stream);
}

} // extern "C"
