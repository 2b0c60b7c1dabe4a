#include "Staging.h"

#include <algorithm>
#include <cfenv>
#include <chrono>
#include <cmath>
#include <cstring>
#include <fstream>
#include <string>

#if defined(__linux__)
#include <sched.h>
#endif
#if defined(__x86_64__)
#include <immintrin.h>
#endif

namespace glow_mi355x {

namespace {

inline void cpuRelax() {
#if defined(__x86_64__)
  _mm_pause();
#endif
}

// The copies below leave the caches out (the device reads the bytes next, over PCIe: 64
// float images 1350 us with ordinary stores, 1315 with these); what they stored is in
// order with what follows only behind this.
inline void storesDone() {
#if defined(__x86_64__)
  _mm_sfence();
#endif
}

// d[i] = s[i] for n int64 values; false when one of them does not fit 32 bits.
bool narrowScalar(int32_t *d, const int64_t *s, size_t n) {
  int64_t bad = 0;
  for (size_t i = 0; i < n; i++) {
    d[i] = (int32_t)s[i];
    bad |= s[i] ^ (int64_t)d[i];
  }
  return bad == 0;
}

#if defined(__x86_64__)
__attribute__((target("avx2"))) bool narrowAvx2(int32_t *d, const int64_t *s, size_t n) {
  __m256i bad = _mm256_setzero_si256();
  size_t i = 0;
  for (; i + 8 <= n; i += 8) {
    const __m256i a = _mm256_loadu_si256((const __m256i *)(s + i));
    const __m256i b = _mm256_loadu_si256((const __m256i *)(s + i + 4));
    // low and high words of the eight values; a high word is the sign of the low one
    const __m256 fa = _mm256_castsi256_ps(a), fb = _mm256_castsi256_ps(b);
    const __m256i lo = _mm256_castps_si256(_mm256_shuffle_ps(fa, fb, 0x88));
    const __m256i hi = _mm256_castps_si256(_mm256_shuffle_ps(fa, fb, 0xdd));
    bad = _mm256_or_si256(bad, _mm256_xor_si256(hi, _mm256_srai_epi32(lo, 31)));
    _mm256_stream_si256((__m256i *)(d + i), _mm256_permute4x64_epi64(lo, 0xd8));
  }
  return _mm256_testz_si256(bad, bad) && narrowScalar(d + i, s + i, n - i);
}
#endif

// The low 16 bits of n int64 values to `low`, past the caches, the next eight to `high`;
// returns the values' OR (what they have to fit in for either to be enough).
uint64_t splitScalar(uint16_t *low, uint8_t *high, const int64_t *s, size_t n) {
  uint64_t all = 0;
  for (size_t i = 0; i < n; i++) {
    low[i] = (uint16_t)s[i];
    high[i] = (uint8_t)(s[i] >> 16);
    all |= (uint64_t)s[i];
  }
  return all;
}

#if defined(__x86_64__)
__attribute__((target("avx2"))) uint64_t splitAvx2(uint16_t *low, uint8_t *high, const int64_t *s,
                                                   size_t n) {
  const __m256i low16 = _mm256_set1_epi32(0xffff), zero = _mm256_setzero_si256();
  __m256i all = zero;
  size_t i = 0;
  for (; i + 16 <= n; i += 16) {
    __m256i x[4], lo[2];
    for (int k = 0; k < 4; k++) {
      x[k] = _mm256_loadu_si256((const __m256i *)(s + i + 4 * k));
      all = _mm256_or_si256(all, x[k]);
    }
    for (int k = 0; k < 2; k++)   // the low words of eight values, in order
      lo[k] = _mm256_permute4x64_epi64(
          _mm256_castps_si256(_mm256_shuffle_ps(_mm256_castsi256_ps(x[2 * k]),
                                                _mm256_castsi256_ps(x[2 * k + 1]), 0x88)),
          0xd8);
    const __m256i w = _mm256_packus_epi32(_mm256_and_si256(lo[0], low16), _mm256_and_si256(lo[1], low16));
    _mm256_stream_si256((__m256i *)(low + i), _mm256_permute4x64_epi64(w, 0xd8));
    // (values of 2^24 and more saturate here; their piece is sent another way)
    const __m256i h = _mm256_permute4x64_epi64(
        _mm256_packus_epi32(_mm256_srli_epi32(lo[0], 16), _mm256_srli_epi32(lo[1], 16)), 0xd8);
    _mm_storeu_si128((__m128i *)(high + i),
                     _mm256_castsi256_si128(_mm256_permute4x64_epi64(_mm256_packus_epi16(h, zero), 0x08)));
  }
  uint64_t part[4];
  _mm256_storeu_si256((__m256i *)part, all);
  return part[0] | part[1] | part[2] | part[3] | splitScalar(low + i, high + i, s + i, n - i);
}
#endif

uint64_t split(uint16_t *low, uint8_t *high, const int64_t *s, size_t n) {
#if defined(__x86_64__)
  static const bool avx2 = __builtin_cpu_supports("avx2");
  if (avx2) return splitAvx2(low, high, s, n);
#endif
  return splitScalar(low, high, s, n);
}

// The high bytes of n values to where the device reads them, as they are or, all below
// 16, two to a byte.
void highBytesScalar(uint8_t *d, const uint8_t *high, size_t n, bool halves) {
  if (!halves) {
    std::memcpy(d, high, n);
    return;
  }
  for (size_t i = 0; i < n; i += 2)
    d[i / 2] = (uint8_t)(high[i] | (i + 1 < n ? high[i + 1] << 4 : 0));
}

#if defined(__x86_64__)
__attribute__((target("avx2"))) void highBytesAvx2(uint8_t *d, const uint8_t *high, size_t n,
                                                   bool halves) {
  const __m256i weights = _mm256_set1_epi16(0x1001);
  size_t i = 0;
  if (halves) {
    for (; i + 32 <= n; i += 32) {
      const __m256i x = _mm256_maddubs_epi16(_mm256_loadu_si256((const __m256i *)(high + i)), weights);
      const __m256i p = _mm256_permute4x64_epi64(_mm256_packus_epi16(x, x), 0x08);
      _mm_stream_si128((__m128i *)(d + i / 2), _mm256_castsi256_si128(p));
    }
    highBytesScalar(d + i / 2, high + i, n - i, true);
  } else {
    for (; i + 32 <= n; i += 32)
      _mm_stream_si128((__m128i *)(d + i), _mm_loadu_si128((const __m128i *)(high + i))),
          _mm_stream_si128((__m128i *)(d + i + 16), _mm_loadu_si128((const __m128i *)(high + i + 16)));
    highBytesScalar(d + i, high + i, n - i, false);
  }
}
#endif

void highBytes(uint8_t *d, const uint8_t *high, size_t n, bool halves) {
#if defined(__x86_64__)
  static const bool avx2 = __builtin_cpu_supports("avx2");
  if (avx2) return highBytesAvx2(d, high, n, halves);
#endif
  highBytesScalar(d, high, n, halves);
}

// n bag lengths as a byte each; false when one of them does not fit.
bool lengthBytesScalar(uint8_t *d, const uint8_t *s, size_t n) {
  uint32_t all = 0;
  for (size_t i = 0; i < n; i++) {
    uint32_t v;
    std::memcpy(&v, s + 4 * i, 4);
    all |= v;
    d[i] = (uint8_t)v;
  }
  return all < 256;
}

#if defined(__x86_64__)
__attribute__((target("avx2"))) bool lengthBytesAvx2(uint8_t *d, const uint8_t *s, size_t n) {
  const __m256i order = _mm256_setr_epi32(0, 4, 1, 5, 2, 6, 3, 7);
  __m256i all = _mm256_setzero_si256();
  size_t i = 0;
  for (; i + 32 <= n; i += 32) {
    __m256i x[4];
    for (int k = 0; k < 4; k++) {
      x[k] = _mm256_loadu_si256((const __m256i *)(s + 4 * (i + 8 * k)));
      all = _mm256_or_si256(all, x[k]);
    }
    // (what does not fit saturates; such lengths are sent another way)
    const __m256i p = _mm256_packus_epi16(_mm256_packus_epi32(x[0], x[1]), _mm256_packus_epi32(x[2], x[3]));
    _mm256_stream_si256((__m256i *)(d + i), _mm256_permutevar8x32_epi32(p, order));
  }
  return _mm256_testz_si256(all, _mm256_set1_epi32(~0xff)) &&
         lengthBytesScalar(d + i, s + 4 * i, n - i);
}
#endif

bool lengthBytes(uint8_t *d, const uint8_t *s, size_t n) {
#if defined(__x86_64__)
  static const bool avx2 = __builtin_cpu_supports("avx2");
  if (avx2) return lengthBytesAvx2(d, s, n);
#endif
  return lengthBytesScalar(d, s, n);
}

// Quantize as the device kernel does it: clip((int32)rint(x / scale + offset)), IEEE
// division, round to even, values past int32 saturating and NaN giving zero.
void quantizeScalar(int8_t *d, const uint8_t *s, size_t n, float scale, float offset) {
  for (size_t i = 0; i < n; i++) {
    float x;
    std::memcpy(&x, s + 4 * i, 4);
    const float r = std::nearbyint(x / scale + offset);
    d[i] = r != r ? 0 : (int8_t)std::max(-128.0f, std::min(127.0f, r));
  }
}

#if defined(__x86_64__)
__attribute__((target("avx2"))) void quantizeAvx2(int8_t *d, const uint8_t *s, size_t n, float scale,
                                                  float offset) {
  const __m256 vs = _mm256_set1_ps(scale), vo = _mm256_set1_ps(offset);
  const __m256 lo = _mm256_set1_ps(-200.0f), hi = _mm256_set1_ps(200.0f);
  const __m256i order = _mm256_setr_epi32(0, 4, 1, 5, 2, 6, 3, 7);
  size_t i = 0;
  for (; i + 32 <= n; i += 32) {
    __m256i r[4];
    for (int k = 0; k < 4; k++) {
      __m256 x = _mm256_loadu_ps((const float *)(s + 4 * (i + 8 * k)));
      x = _mm256_add_ps(_mm256_div_ps(x, vs), vo);
      x = _mm256_and_ps(x, _mm256_cmp_ps(x, x, _CMP_ORD_Q));   // NaN -> 0
      r[k] = _mm256_cvtps_epi32(_mm256_min_ps(_mm256_max_ps(x, lo), hi));
    }
    const __m256i q = _mm256_packs_epi16(_mm256_packs_epi32(r[0], r[1]), _mm256_packs_epi32(r[2], r[3]));
    _mm256_stream_si256((__m256i *)(d + i), _mm256_permutevar8x32_epi32(q, order));
  }
  quantizeScalar(d + i, s + 4 * i, n - i, scale, offset);
}
#endif

// The rounding mode and the treatment of denormals that the kernel has, whichever
// thread takes a piece: the caller's are its own, and threads start with those of the
// one that made them.
class DefaultFloats {
public:
#if defined(__x86_64__)
  DefaultFloats() : kept_(_mm_getcsr()) { _mm_setcsr(0x1f80); }
  ~DefaultFloats() { _mm_setcsr(kept_); }

private:
  unsigned kept_;
#else
  DefaultFloats() { std::fegetenv(&kept_), std::fesetenv(FE_DFL_ENV); }
  ~DefaultFloats() { std::fesetenv(&kept_); }

private:
  std::fenv_t kept_;
#endif
};

__attribute__((noinline)) void quantizeDefault(int8_t *d, const uint8_t *s, size_t n, float scale,
                                               float offset) {
#if defined(__x86_64__)
  static const bool avx2 = __builtin_cpu_supports("avx2");
  if (avx2) return quantizeAvx2(d, s, n, scale, offset);
#endif
  quantizeScalar(d, s, n, scale, offset);
}

void quantize(int8_t *d, const uint8_t *s, size_t n, float scale, float offset) {
  const DefaultFloats floats;
  quantizeDefault(d, s, n, scale, offset);
}

bool narrow(int32_t *d, const int64_t *s, size_t n) {
#if defined(__x86_64__)
  static const bool avx2 = __builtin_cpu_supports("avx2");
  if (avx2) return narrowAvx2(d, s, n);
#endif
  return narrowScalar(d, s, n);
}

} // namespace

namespace {

// The quota of one control group in CPUs (cpu.max: "quota period", or "max"); 0 = none.
int groupCpus(const std::string &dir) {
  std::ifstream v2(dir + "/cpu.max"), v1(dir + "/cpu.cfs_quota_us"), v1p(dir + "/cpu.cfs_period_us");
  double quota = 0, period = 0;
  if (v2 ? !(v2 >> quota >> period) : !(v1 >> quota && v1p >> period)) return 0;
  return quota > 0 && period > 0 ? std::max(1, (int)(quota / period)) : 0;
}

// CPUs this process may use: those it may be scheduled on, within the quotas of the
// control groups it is in (a container's share of a larger machine).
int cpusToUse() {
  int n = (int)std::thread::hardware_concurrency();
#if defined(__linux__)
  cpu_set_t set;
  if (sched_getaffinity(0, sizeof set, &set) == 0) n = CPU_COUNT(&set);
  auto within = [&](const std::string &dir) {
    const int q = groupCpus(dir);
    if (q > 0) n = std::min(n, q);
  };
  std::ifstream groups("/proc/self/cgroup");   // "id:controllers:/path", one a hierarchy
  for (std::string line; std::getline(groups, line);) {
    const size_t a = line.find(':'), b = a == std::string::npos ? a : line.find(':', a + 1);
    if (b == std::string::npos) continue;
    const std::string controllers = line.substr(a + 1, b - a - 1);
    std::string root = "/sys/fs/cgroup", path = line.substr(b + 1);
    if (!controllers.empty()) {
      if (("," + controllers + ",").find(",cpu,") == std::string::npos) continue;
      root += "/cpu";
    }
    if (path.empty() || path[0] != '/') continue;
    for (; path.size() > 1; path.resize(path.rfind('/'))) within(root + path);
    within(root);
  }
#endif
  return std::max(1, n);
}

// A third of them, for helpers: of one pool, and of all pools together for those that
// are awake without work.
int helperCpus() {
  static const int n = cpusToUse() / 3;
  return n;
}
std::atomic<int> g_awake{0};

} // namespace

StagingPool::StagingPool() {
  // five at most: a batch of 64 float images (38.5 MB, quantized) takes 1610 us with two
  // helpers, 1500 with three, 1410, 1350 with five, 1335 with seven or eleven
  for (int i = 0; i < std::min(5, helperCpus()); i++) threads_.emplace_back([this] { loop(); });
}

StagingPool::~StagingPool() {
  {
    std::lock_guard<std::mutex> lk(mu_);
    stopping_ = true;
    generation_++;
  }
  cv_.notify_all();
  for (auto &t : threads_) t.join();
}

void StagingPool::stage(StagePiece &p, uint8_t *buffer) {
  uint8_t *d = buffer + p.at;
  p.seg.src = d;
  p.seg.bytes = p.bytes;
  if (p.form == StagePiece::Quantized) {
    quantize((int8_t *)d, p.src, p.bytes / 4, p.scale, p.offset);
    storesDone();
    p.seg.bytes = p.bytes / 4;
    return;
  }
  if (p.form == StagePiece::Lengths) {
    const bool packed = lengthBytes(d, p.src, p.bytes / 4);
    storesDone();
    if (packed) {
      p.seg.op = MI355X_SEGMENT_LENGTHS_U8;
      p.seg.bytes = p.bytes / 4;
      return;
    }
  }
  if (p.form == StagePiece::Indices64 && ((uintptr_t)p.src & 7) == 0) {
    // the fewest bytes a value that hold all of the piece
    const int64_t *v = (const int64_t *)p.src;
    const size_t n = p.bytes / 8, plane = (2 * n + 15) & ~(size_t)15;
    // (the high bytes are looked at once more before they are stored)
    uint8_t high[kStagePiece / 8];
    const uint64_t all =
        plane + n <= p.bytes && n <= sizeof high ? split((uint16_t *)d, high, v, n) : ~(uint64_t)0;
    if (all < (1u << 24)) {
      const bool halves = all < (1u << 20);
      p.seg.op = all < (1u << 16) ? MI355X_SEGMENT_WIDEN_U16
                 : halves         ? MI355X_SEGMENT_WIDEN_U20
                                  : MI355X_SEGMENT_WIDEN_U24;
      if (all >= (1u << 16)) highBytes(d + plane, high, n, halves);
      storesDone();
      p.seg.bytes = 2 * n;
      return;
    }
    storesDone();
    const bool narrowed = narrow((int32_t *)d, v, n);
    storesDone();
    if (narrowed) {
      p.seg.op = MI355X_SEGMENT_WIDEN_I32;
      p.seg.bytes = 4 * n;
      return;
    }
  }
  std::memcpy(d, p.src, p.bytes);
}

void StagingPool::open(std::vector<StagePiece> &pieces, uint8_t *buffer, bool wake) {
  if (room_ < pieces.size()) {
    room_ = pieces.size();
    done_.reset(new std::atomic<uint8_t>[room_]);
  }
  for (size_t i = 0; i < pieces.size(); i++) done_[i].store(0, std::memory_order_relaxed);
  std::lock_guard<std::mutex> lk(mu_);
  pieces_ = pieces.data();
  buffer_ = buffer;
  count_ = pieces.size();
  next_ = 0;
  if (wake) {
    openJob_ = true;
    generation_++;
    cv_.notify_all();
  }
}

void StagingPool::close() {
  {
    std::lock_guard<std::mutex> lk(mu_);
    openJob_ = false;
  }
  while (active_.load(std::memory_order_acquire) != 0) cpuRelax();
}

void StagingPool::work() {
  for (;;) {
    const size_t i = next_.fetch_add(1, std::memory_order_relaxed);
    if (i >= count_) return;
    stage(pieces_[i], buffer_);
    done_[i].store(1, std::memory_order_release);
  }
}

void StagingPool::loop() {
  uint64_t seen = 0;
  for (;;) {
    // a moment awake between jobs: the next request of a busy server is there
    // before a sleeping thread would be (waking one takes some 50 us; a ranking request of
    // 4096 samples 322 us when they wait 100 us for the next, 309 at 500, 310 at 2000).
    // Beyond a third of the CPUs, with several managers in one process, they sleep at once.
    if (g_awake.fetch_add(1, std::memory_order_relaxed) < helperCpus()) {
      const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(500);
      while (generation_.load(std::memory_order_acquire) == seen &&
             std::chrono::steady_clock::now() < until)
        for (int i = 0; i < 16; i++) cpuRelax();
    }
    g_awake.fetch_sub(1, std::memory_order_relaxed);
    {
      std::unique_lock<std::mutex> lk(mu_);
      cv_.wait(lk, [&] { return generation_.load() != seen; });
      seen = generation_;
      if (stopping_) return;
      if (!openJob_) continue;
      active_.fetch_add(1, std::memory_order_relaxed);
    }
    work();
    active_.fetch_sub(1, std::memory_order_release);
  }
}

} // namespace glow_mi355x
