// Many small transfers in one launch: the inputs of a request out of pinned host
// memory into their slots, and its outputs back. A copy queued on the DMA engines
// costs 10 to 20 us whatever its size, so the 54 inputs of a 26-table ranking
// request took 1.1 ms for 17 MB; compute units that read the pinned memory
// themselves over PCIe move the same bytes at 50 GB/s in one launch.
#include "common.h"

namespace mi355x {

constexpr int kSegThreads = 256;
constexpr int kSegInFlight = 4;   // 16-byte requests of a thread in flight
// 16 KiB per workgroup: a request of 64 KiB is spread over four CUs, and 17 MB
// are a thousand workgroups, 4 KiB of requests in flight each (the PCIe link
// needs 0.1 MB in flight).
constexpr uint32_t kSegBlockBytes = kSegThreads * 16 * kSegInFlight;
constexpr int kSegMax = 64;       // descriptors per launch: 2.5 KB of arguments
constexpr int kLengthsPerThread = 16;

struct SegArg {
  uint8_t *dst;
  const uint8_t *src;
  int32_t *positions;
  uint32_t bytes;        // of src
  uint32_t first_block;
  uint32_t op;
  uint32_t count;        // LENGTHS: bags of the placeholder
};
struct SegArgs {
  SegArg seg[kSegMax];
  int n;
  uint32_t done_value;
  uint32_t *done;        // host memory, NULL = nobody waits
  uint32_t *arrived;     // device counter, zero between launches
};

__device__ __forceinline__ void seg_copy(const SegArg &s, uint32_t at, uint32_t end, int tid) {
  const bool vec = ((((uintptr_t)s.dst) | ((uintptr_t)s.src)) & 15) == 0;
  uint32_t i = at;
  if (vec) {
    // (all of a thread's loads in flight, in a part of a block too: a trip over the
    // link takes 2 us)
    const uint32_t pieces = (end - at) / 16;
    const int4 *p = reinterpret_cast<const int4 *>(s.src + at);
    int4 *q = reinterpret_cast<int4 *>(s.dst + at);
    int4 v[kSegInFlight];
#pragma unroll
    for (uint32_t u = 0; u < kSegInFlight; u++)
      if (tid + u * kSegThreads < pieces) v[u] = p[tid + u * kSegThreads];
#pragma unroll
    for (uint32_t u = 0; u < kSegInFlight; u++)
      if (tid + u * kSegThreads < pieces) q[tid + u * kSegThreads] = v[u];
    i += pieces * 16;
  }
  for (i += tid; i < end; i += kSegThreads) s.dst[i] = s.src[i];
}

// int32 on the wire, int64 in the slot (16-byte aligned both; whole int32s)
__device__ __forceinline__ void seg_widen(const SegArg &s, uint32_t at, uint32_t end, int tid) {
  auto put = [&](uint32_t i, const int4 &v) {
    longlong2 *q = reinterpret_cast<longlong2 *>(s.dst + 2 * (size_t)i);
    q[0] = make_longlong2(v.x, v.y);
    q[1] = make_longlong2(v.z, v.w);
  };
  const uint32_t pieces = (end - at) / 16, whole = at + pieces * 16;
  const int4 *p = reinterpret_cast<const int4 *>(s.src + at);
  int4 v[kSegInFlight];
#pragma unroll
  for (uint32_t u = 0; u < kSegInFlight; u++)
    if (tid + u * kSegThreads < pieces) v[u] = p[tid + u * kSegThreads];
#pragma unroll
  for (uint32_t u = 0; u < kSegInFlight; u++)
    if (tid + u * kSegThreads < pieces) put(at + (tid + u * kSegThreads) * 16, v[u]);
  for (uint32_t i = whole + tid * 4; i < end; i += kSegThreads * 4)
    *reinterpret_cast<long long *>(s.dst + 2 * (size_t)i) = *reinterpret_cast<const int32_t *>(s.src + i);
}

// 16 bits, or 16 and HIGH = 4 or 8 in two planes, on the wire, int64 in the slot. The
// planes pass through LDS: 16-byte loads and 16-byte stores of neighbouring lanes to
// neighbouring places. The PCIe link
// bounds a request of indices, 20 us per MB: at 4096 samples of 26 x 20 lookups three
// bytes a value instead of four 381 us a request before, 322 then (two bytes: 376, 278);
// two and a half instead of three, with the lengths in a byte each, 313 before, 296 then.
template <int HIGH>
__device__ __forceinline__ void seg_widen_planes(const SegArg &s, uint32_t at, uint32_t end, int tid) {
  __shared__ __attribute__((aligned(16))) uint32_t s_low[kSegBlockBytes / 4];
  __shared__ __attribute__((aligned(16))) uint8_t s_high[kSegBlockBytes / 2];   // a byte a value at most
  const int bytes = (int)(end - at), n = bytes / 2;
  const uint8_t *low = s.src + at;
  const uint8_t *high = s.src + (((size_t)s.bytes + 15) & ~(size_t)15) + (size_t)at / 2 * HIGH / 8;
  const int high_bytes = (n * HIGH + 7) / 8;
  long long *out = reinterpret_cast<long long *>(s.dst) + at / 2;
  // (a part of a block the same way: value by value it took 50 us of trips over the link)
  constexpr int kHighLoads = HIGH == 8 ? kSegInFlight / 2 : kSegInFlight / 4;
  int4 v[kSegInFlight], h[kHighLoads];
#pragma unroll
  for (int u = 0; u < kSegInFlight; u++) {
    const int i = tid + u * kSegThreads;
    if (i < bytes / 16) v[u] = reinterpret_cast<const int4 *>(low)[i];
  }
  if constexpr (HIGH != 0) {
#pragma unroll
    for (int u = 0; u < kHighLoads; u++) {
      const int i = tid + u * kSegThreads;
      if (i < high_bytes / 16) h[u] = reinterpret_cast<const int4 *>(high)[i];
    }
  }
  const int last = n / 8 * 8 + tid, last_high = high_bytes / 16 * 16 + tid;   // what is no whole load
  if (last < n) reinterpret_cast<uint16_t *>(s_low)[last] = reinterpret_cast<const uint16_t *>(low)[last];
  if (HIGH != 0 && last_high < high_bytes) s_high[last_high] = high[last_high];
#pragma unroll
  for (int u = 0; u < kSegInFlight; u++) {
    const int i = tid + u * kSegThreads;
    if (i < bytes / 16) reinterpret_cast<int4 *>(s_low)[i] = v[u];
  }
  if constexpr (HIGH != 0) {
#pragma unroll
    for (int u = 0; u < kHighLoads; u++) {
      const int i = tid + u * kSegThreads;
      if (i < high_bytes / 16) reinterpret_cast<int4 *>(s_high)[i] = h[u];
    }
  }
  __syncthreads();
  for (int p = tid; p < (n + 1) / 2; p += kSegThreads) {
    const uint32_t w = s_low[p];
    uint32_t a = w & 0xffff, b = w >> 16;
    if constexpr (HIGH == 8) {
      const uint32_t t = reinterpret_cast<const uint16_t *>(s_high)[p];
      a |= (t & 0xff) << 16;
      b |= (t & 0xff00) << 8;
    } else if constexpr (HIGH == 4) {
      const uint32_t t = s_high[p];
      a |= (t & 0xf) << 16;
      b |= (t & 0xf0) << 12;
    }
    if (2 * p + 1 < n) reinterpret_cast<longlong2 *>(out)[p] = make_longlong2(a, b);
    else out[2 * p] = a;
  }
}

// Lengths of bags: copied, the rest of the slot cleared, and the positions
// (exclusive prefix sums of the lengths, negative ones counting as empty bags,
// saturating at INT32_MAX) written; one workgroup, sixteen lengths per thread and
// round, all of a round's loads in one trip. BYTES: a byte each on the wire.
template <bool BYTES>
__device__ __forceinline__ void seg_lengths(const SegArg &s, int tid) {
  __shared__ long long s_wave[kSegThreads / 64];
  const int32_t *src = reinterpret_cast<const int32_t *>(s.src);
  int32_t *dst = reinterpret_cast<int32_t *>(s.dst);
  const int n = BYTES ? (int)s.bytes : (int)(s.bytes / 4), bags = (int)s.count;
  const int lane = tid & 63, wave = tid >> 6;
  const bool vec = (((uintptr_t)src) & 15) == 0;
  long long carry = 0;
  for (int base = 0; base < bags; base += kSegThreads * kLengthsPerThread) {
    const int i0 = base + tid * kLengthsPerThread;
    int v[kLengthsPerThread];
    if (vec && i0 + kLengthsPerThread <= n) {
      if constexpr (BYTES) {
        static_assert(kLengthsPerThread == 16, "one load a thread");
        const int4 x = *reinterpret_cast<const int4 *>(s.src + i0);
        const uint32_t w[4] = {(uint32_t)x.x, (uint32_t)x.y, (uint32_t)x.z, (uint32_t)x.w};
#pragma unroll
        for (int u = 0; u < 16; u++) v[u] = (int)((w[u / 4] >> (8 * (u % 4))) & 0xff);
      } else {
#pragma unroll
        for (int u = 0; u < kLengthsPerThread / 4; u++) {
          const int4 x = *reinterpret_cast<const int4 *>(src + i0 + 4 * u);
          v[4 * u] = x.x; v[4 * u + 1] = x.y; v[4 * u + 2] = x.z; v[4 * u + 3] = x.w;
        }
      }
    } else {
#pragma unroll
      for (int u = 0; u < kLengthsPerThread; u++)
        v[u] = i0 + u >= n ? 0 : BYTES ? (int)s.src[i0 + u] : src[i0 + u];
    }
    long long mine = 0;
#pragma unroll
    for (int u = 0; u < kLengthsPerThread; u++) mine += max(v[u], 0);
    long long incl = mine;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const long long below = __shfl_up(incl, off, 64);
      if (lane >= off) incl += below;
    }
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    long long at = carry + incl - mine;
#pragma unroll
    for (int w = 0; w < kSegThreads / 64; w++) {
      if (w < wave) at += s_wave[w];
      carry += s_wave[w];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kLengthsPerThread; u++) {
      if (i0 + u < bags) {
        if (dst) dst[i0 + u] = v[u];
        s.positions[i0 + u] = (int32_t)min(at, 0x7fffffffLL);
        at += max(v[u], 0);
      }
    }
  }
  if (tid == 0) s.positions[bags] = (int32_t)min(carry, 0x7fffffffLL);
}

__global__ __launch_bounds__(kSegThreads) void copy_segments_kernel(SegArgs a) {
  const int tid = threadIdx.x;
  int lo = 0, hi = a.n - 1;          // the last segment that starts at or before this block
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (a.seg[mid].first_block <= blockIdx.x) lo = mid;
    else hi = mid - 1;
  }
  const SegArg s = a.seg[lo];
  const uint32_t at = (blockIdx.x - s.first_block) * kSegBlockBytes;
  const uint32_t end = min(s.bytes, at + kSegBlockBytes);
  if (s.op == MI355X_SEGMENT_LENGTHS) seg_lengths<false>(s, tid);
  else if (s.op == MI355X_SEGMENT_LENGTHS_U8) seg_lengths<true>(s, tid);
  else if (s.op == MI355X_SEGMENT_WIDEN_I32) seg_widen(s, at, end, tid);
  else if (s.op == MI355X_SEGMENT_WIDEN_U16) seg_widen_planes<0>(s, at, end, tid);
  else if (s.op == MI355X_SEGMENT_WIDEN_U20) seg_widen_planes<4>(s, at, end, tid);
  else if (s.op == MI355X_SEGMENT_WIDEN_U24) seg_widen_planes<8>(s, at, end, tid);
  else seg_copy(s, at, end, tid);
  if (a.done) {
    // the block that arrives last tells the host; every block's stores have
    // reached it by then
    __threadfence_system();
    __syncthreads();
    if (tid == 0 &&
        __hip_atomic_fetch_add(a.arrived, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) ==
            gridDim.x - 1) {
      __hip_atomic_store(a.arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(a.done, a.done_value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

} // namespace mi355x

using namespace mi355x;

extern "C" {

int mi355x_copy_segments(const mi355x_copy_segment *segments, size_t n, uint32_t *done,
                         uint32_t done_value, uint32_t *arrived, void *stream) {
  MI355X_REQUIRE(segments || n == 0, "segments is NULL");
  MI355X_REQUIRE(!done || (arrived && n > 0), "a done flag needs a counter and a segment");
  SegArgs a{};
  uint32_t blocks = 0;
  auto flush = [&](bool last) {
    if (a.n == 0) return (int)MI355X_OK;
    a.done = last ? done : nullptr;
    a.done_value = done_value;
    a.arrived = arrived;
    hipLaunchKernelGGL(copy_segments_kernel, dim3(blocks), dim3(kSegThreads), 0, as_stream(stream), a);
    a.n = 0;
    blocks = 0;
    return check_launch("copy_segments");
  };
  for (size_t i = 0; i < n; i++) {
    const mi355x_copy_segment &s = segments[i];
    const bool lengths = s.op == MI355X_SEGMENT_LENGTHS || s.op == MI355X_SEGMENT_LENGTHS_U8;
    MI355X_REQUIRE(s.op >= MI355X_SEGMENT_COPY && s.op <= MI355X_SEGMENT_LENGTHS_U8,
                   "unknown segment operation %d", s.op);
    MI355X_REQUIRE(s.bytes < (1ull << 31), "segment of %llu bytes: at most 2^31 - 1",
                   (unsigned long long)s.bytes);
    MI355X_REQUIRE((s.src || s.bytes == 0) && (s.dst || lengths),
                   "NULL segment");
    if (s.op == MI355X_SEGMENT_WIDEN_I32)
      MI355X_REQUIRE(s.bytes % 4 == 0 && ((((uintptr_t)s.src) | ((uintptr_t)s.dst)) & 15) == 0,
                     "a widened segment is whole int32s at 16-byte boundaries");
    if (s.op == MI355X_SEGMENT_WIDEN_U16 || s.op == MI355X_SEGMENT_WIDEN_U20 ||
        s.op == MI355X_SEGMENT_WIDEN_U24)
      MI355X_REQUIRE(s.bytes % 2 == 0 && ((((uintptr_t)s.src) | ((uintptr_t)s.dst)) & 15) == 0,
                     "a widened segment is whole uint16s at 16-byte boundaries");
    if (s.op == MI355X_SEGMENT_LENGTHS)
      MI355X_REQUIRE(s.positions && s.bags < (1u << 30) && s.bytes % 4 == 0 &&
                         s.bytes / 4 <= s.bags && (((uintptr_t)s.src) & 3) == 0,
                     "lengths segment: %llu bytes for %u bags", (unsigned long long)s.bytes, s.bags);
    if (s.op == MI355X_SEGMENT_LENGTHS_U8)
      MI355X_REQUIRE(s.positions && s.bags < (1u << 30) && s.bytes <= s.bags,
                     "lengths segment: %llu bytes for %u bags", (unsigned long long)s.bytes, s.bags);
    if (a.n == kSegMax) {
      const int rc = flush(false);
      if (rc != MI355X_OK) return rc;
    }
    SegArg &d = a.seg[a.n++];
    d.dst = (uint8_t *)s.dst;
    d.src = (const uint8_t *)s.src;
    d.positions = s.positions;
    d.bytes = (uint32_t)s.bytes;
    d.first_block = blocks;
    d.op = (uint32_t)s.op;
    d.count = s.bags;
    const uint32_t need = (uint32_t)((s.bytes + kSegBlockBytes - 1) / kSegBlockBytes);
    blocks += lengths || need == 0 ? 1 : need;
  }
  return flush(true);
}

} // extern "C"
