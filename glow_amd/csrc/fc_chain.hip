// A chain of RowwiseQuantizedFullyConnected layers in one kernel: the towers of a
// ranking net, each layer reading what the one in front of it wrote. As launches of their
// own such layers are mostly dispatch and trips to memory. Here a workgroup takes sixteen
// rows through all of them: the rows' bytes stay in LDS between the layers, the weights
// pass through registers on their way from L2.
//
// Weights are packed once, when a network is loaded, in the order the matrix cores take
// them: [tile of 16 outputs][step of 64 inputs][lane][16 bytes], zeros where a layer has
// no input or output, so that a wave's load is 1 KB on end whatever K is (rows of 415
// bytes would come by words), and what lies in LDS past a row's end multiplies zeros. They
// are the first operand: a lane's four results are then four neighbouring outputs of one
// row, a word of the next layer's input. The per-column constants (the rescaled bias with
// the input offset's share, shifts and scale) are packed with them.
//
// What bounds it: the dispatch and the trips of the layers in turn, each as long as its
// weights' way from L2 into one compute unit (some 85 bytes per ns with sixteen waves of
// up to 8 KB in flight each; a wave asks for its next tile as soon as it has multiplied one,
// across the barrier into the next layer too). Sixteen rows to a workgroup put 4096 rows on
// every compute unit once. us, layer by layer / chain: 13 -> 512 -> 256 -> 64 over 4096 rows
// 15.3 / 7.9, over 16 rows 11.8 / 7.0; 415 -> 512 -> 256 -> 1 16.6 / 9.1 and 11.9 / 8.3. A ranking
// net's fourteen launches become four: 94 / 68 us of them at batch 4096, 38 / 26 at batch 16.
#include "common.h"
#pragma clang fp contract(off)
#include "requant.h"

namespace mi355x {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kChainRows = 16;                         // rows of a workgroup
constexpr int kChainPitch = MI355X_FC_CHAIN_WIDTH + 16; // of a row in LDS: no bank twice
enum { kColConst, kColPre, kColScale, kColPost, kColArrays };

struct ChainLayer {
  const int8_t *w;
  const int32_t *col;   // [kColArrays][tiles * 16]
  int steps, group, tiles, n;   // steps: a multiple of group (chain_steps)
  int out_off, relu, relu_off, relu_pre, relu_post, relu_scale;
};
struct ChainSlice {
  int8_t *dst;
  long long pitch;
  int out_off, in_off, pre, post, scale;
};
struct ChainArgs {
  ChainLayer layer[MI355X_FC_CHAIN_LAYERS];
  int layers, M, K;
  const int8_t *in;
  const float *in_f32;
  float in_scale, in_offset;
  int8_t *out;
  ChainSlice slice[MI355X_FC_CHAIN_SLICES];
  int slices;
  float *sigmoid;
  float sigmoid_scale;
  int sigmoid_off;
};

struct __attribute__((packed, aligned(1))) AnyWord { uint32_t w; };

// up to four neighbouring bytes of a row, at any address
__device__ __forceinline__ void store_some(int8_t *p, uint32_t word, int n) {
  if (n >= 4) {
    reinterpret_cast<AnyWord *>(p)->w = word;
  } else {
    for (int j = 0; j < n; j++) p[j] = (int8_t)(word >> (8 * j));
  }
}
__device__ __forceinline__ uint32_t pack_bytes(const int32_t (&y)[4]) {
  return (uint32_t)(y[0] & 0xff) | ((uint32_t)(y[1] & 0xff) << 8) | ((uint32_t)(y[2] & 0xff) << 16) |
         ((uint32_t)(y[3] & 0xff) << 24);
}

// The weight fragments of a group of steps, by name and passed by value: as an array they
// end up in scratch memory, because the branches' loads are merged and their targets then
// picked by address (eight times the launch's time).
struct Frags {
  v4i a, b, c, d, e, f, g, h;
};
__device__ __forceinline__ Frags load_group(const int8_t *p, int group) {
  auto at = [&](int u) __attribute__((always_inline)) { return *reinterpret_cast<const v4i *>(p + u * 1024); };
  const v4i none{0, 0, 0, 0};
  Frags r{at(0), none, none, none, none, none, none, none};
  if (group > 1) { r.b = at(1); r.c = at(2); r.d = at(3); }
  if (group > 4) { r.e = at(4); r.f = at(5); r.g = at(6); r.h = at(7); }
  return r;
}
__device__ __forceinline__ v4i multiply_group(Frags w, const int8_t *rows, v4i acc, int group) {
  auto on = [&](v4i x, int u, v4i to) __attribute__((always_inline)) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(x, *reinterpret_cast<const v4i *>(rows + u * 64), to, 0, 0, 0);
  };
  acc = on(w.a, 0, acc);
  if (group > 1) acc = on(w.d, 3, on(w.c, 2, on(w.b, 1, acc)));
  if (group > 4) acc = on(w.h, 7, on(w.g, 6, on(w.f, 5, on(w.e, 4, acc))));
  return acc;
}

template <int W>
__global__ __launch_bounds__(W * 64) void fc_chain_i8_kernel(ChainArgs a) {
  __shared__ __attribute__((aligned(16))) int8_t s_rows[2][kChainRows * kChainPitch];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, part = lane >> 4;
  const int m0 = blockIdx.x * kChainRows, m = m0 + r16;

  // the group that starts at step s of tile t
  auto request = [&](const ChainLayer &q, int t, int s) __attribute__((always_inline)) {
    return load_group(q.w + ((long long)t * q.steps + s) * 1024 + lane * 16, q.group);
  };
  ChainLayer L = a.layer[0];
  Frags f{};
  if (wave < L.tiles) f = request(L, wave, 0);

  // the rows' bytes; rows past M repeat the last one and are not stored
  if (a.in_f32) {
    for (int i = tid; i < kChainRows * a.K; i += W * 64) {
      const int r = i / a.K, k = i - r * a.K;
      const float x = a.in_f32[(long long)min(m0 + r, a.M - 1) * a.K + k];
      s_rows[0][r * kChainPitch + k] = (int8_t)quantize_one(x, a.in_scale, a.in_offset);
    }
  } else {
    const int words = (a.K + 3) >> 2;
    for (int i = tid; i < kChainRows * words; i += W * 64) {
      const int r = i / words, k = 4 * (i - r * words);
      const int8_t *p = a.in + (long long)min(m0 + r, a.M - 1) * a.K;
      uint32_t v = 0;
      if (a.K >= 4) {
        const int at = min(k, a.K - 4);               // the last word ends with the row
        v = reinterpret_cast<const AnyWord *>(p + at)->w >> (8 * (k - at));
      } else {
        for (int b = 0; b < a.K; b++) v |= (uint32_t)(uint8_t)p[b] << (8 * b);
      }
      *reinterpret_cast<uint32_t *>(&s_rows[0][r * kChainPitch + k]) = v;
    }
  }
  __syncthreads();

  for (int l = 0; l < a.layers; l++) {
    const bool last = l + 1 == a.layers;
    const ChainLayer next = a.layer[last ? l : l + 1];   // asked for a layer ahead
    const int8_t *src = s_rows[l & 1] + r16 * kChainPitch + part * 16;
    int8_t *dst = s_rows[(l & 1) ^ 1] + r16 * kChainPitch + part * 4;
    const int padded = L.tiles * 16;
    for (int t = wave; t < L.tiles; t += W) {
      const int n = t * 16 + part * 4;
      const int32_t *col = L.col + n;
      const v4i colc = *reinterpret_cast<const v4i *>(col + kColConst * padded);
      const v4i pre = *reinterpret_cast<const v4i *>(col + kColPre * padded);
      const v4i scale = *reinterpret_cast<const v4i *>(col + kColScale * padded);
      const v4i post = *reinterpret_cast<const v4i *>(col + kColPost * padded);
      v4i acc{0, 0, 0, 0};
      for (int s = 0;;) {
        acc = multiply_group(f, src + s * 64, acc, L.group);
        s += L.group;
        if (s >= L.steps) break;
        f = request(L, t, s);
      }
      // what this wave multiplies next travels while these results are requantised and
      // the other waves are waited for
      const bool more = t + W < L.tiles;
      if (more || (!last && wave < next.tiles)) f = request(more ? L : next, more ? t + W : wave, 0);
      int32_t y[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        y[j] = clip_i8(scale_i32((int32_t)((uint32_t)acc[j] + (uint32_t)colc[j]), pre[j], post[j],
                                 scale[j], L.out_off));
        if (L.relu)
          y[j] = clip_i8(scale_i32(max(y[j], L.out_off) - L.out_off, L.relu_pre, L.relu_post,
                                   L.relu_scale, L.relu_off));
      }
      const uint32_t word = pack_bytes(y);
      if (!last) {
        *reinterpret_cast<uint32_t *>(dst + t * 16) = word;
      } else if (m < a.M && n < L.n) {
        const int some = min(4, L.n - n);
        if (a.out) store_some(a.out + (long long)m * L.n + n, word, some);
        for (int q = 0; q < a.slices; q++) {
          const ChainSlice &S = a.slice[q];
          int32_t z[4];
#pragma unroll
          for (int j = 0; j < 4; j++)
            z[j] = clip_i8(scale_i32(y[j] - S.in_off, S.pre, S.post, S.scale, S.out_off));
          store_some(S.dst + m * S.pitch + n, pack_bytes(z), some);
        }
        if (a.sigmoid)
          for (int j = 0; j < 4; j++)
            if (j < some)
              a.sigmoid[(long long)m * L.n + n + j] =
                  sigmoid_of((int8_t)(word >> (8 * j)), a.sigmoid_scale, a.sigmoid_off);
      }
    }
    // a wave without a tile here may have one in the next layer
    if (!last && wave >= L.tiles && wave < next.tiles) f = request(next, wave, 0);
    __syncthreads();
    L = next;
  }
}

// Whether one of `rows` rows of `bytes` bytes, `pitch` apart, lies in [at, at + size).
static bool rows_touch(const void *first, long long pitch, long long rows, long long bytes,
                       const void *at, long long size) {
  const long long off = (long long)((uintptr_t)first - (uintptr_t)at);   // of row 0
  if (bytes == 0 || size == 0 || off >= size) return false;
  // the first row that ends behind `at`
  long long r = 0;
  if (off + bytes <= 0) {
    if (pitch == 0) return false;
    r = (-off - bytes) / pitch + 1;
  }
  return r < rows && off + r * pitch < size;
}

} // namespace mi355x

using namespace mi355x;

extern "C" int mi355x_rwq_fc_chain_i8(const mi355x_fc_chain *c, void *stream) {
  MI355X_REQUIRE(c && c->struct_size == sizeof(mi355x_fc_chain), "struct_size is not this library's");
  MI355X_REQUIRE(c->n_layers >= 1 && c->n_layers <= MI355X_FC_CHAIN_LAYERS, "%d layers", c->n_layers);
  MI355X_REQUIRE(c->n_slices >= 0 && c->n_slices <= MI355X_FC_CHAIN_SLICES, "%d slices", c->n_slices);
  if (c->M == 0) return MI355X_OK;
  MI355X_REQUIRE(c->M < (1u << 30), "too many rows");
  MI355X_REQUIRE(c->in || c->in_f32, "NULL input");
  ChainArgs a{};
  a.layers = c->n_layers;
  a.M = (int)c->M;
  a.in = c->in;
  a.in_f32 = c->in ? nullptr : c->in_f32;
  a.in_scale = c->in_scale;
  a.in_offset = (float)c->in_offset;
  for (int l = 0; l < a.layers; l++) {
    const mi355x_fc_chain_layer &q = c->layers[l];
    MI355X_REQUIRE(q.weights && q.columns, "layer %d: NULL tensor", l);
    MI355X_REQUIRE((((uintptr_t)q.weights | (uintptr_t)q.columns) & 15) == 0,
                   "layer %d: packed constants do not start on 16 bytes", l);
    MI355X_REQUIRE(q.K >= 1 && q.K <= MI355X_FC_CHAIN_WIDTH && q.N >= 1 && q.N <= MI355X_FC_CHAIN_WIDTH,
                   "layer %d: %zu x %zu outside [1, %d]", l, q.K, q.N, MI355X_FC_CHAIN_WIDTH);
    MI355X_REQUIRE(l == 0 || q.K == c->layers[l - 1].N, "layer %d reads %zu values of %zu", l, q.K,
                   l ? c->layers[l - 1].N : 0);
    MI355X_REQUIRE(!q.relu || (shift_ok(q.relu_pre) && shift_ok(q.relu_post)),
                   "relu pre/post shift outside [0, 31]");
    MI355X_REQUIRE(!q.relu || (q.fc_offset >= -128 && q.fc_offset <= 127),
                   "offset %d of the FullyConnected result outside the int8 range", q.fc_offset);
    a.layer[l] = ChainLayer{q.weights, q.columns, chain_steps((int)q.K), chain_group((int)q.K), (int)((q.N + 15) / 16),
                            (int)q.N, q.fc_offset, q.relu, q.relu_offset, q.relu_pre, q.relu_post,
                            q.relu_scale};
  }
  a.K = (int)c->layers[0].K;
  a.out = c->out;
  a.slices = c->n_slices;
  for (int s = 0; s < a.slices; s++) {
    const mi355x_fc_chain_slice &q = c->slices[s];
    MI355X_REQUIRE(q.dst && q.dst_row_stride < (1ull << 40), "slice %d: no destination", s);
    MI355X_REQUIRE(q.dst_row_stride >= c->layers[a.layers - 1].N,
                   "slice %d: rows of %zu bytes overlap at a stride of %zu", s, c->layers[a.layers - 1].N,
                   q.dst_row_stride);
    MI355X_REQUIRE(shift_ok(q.pre) && shift_ok(q.post), "pre/post shift outside [0, 31]");
    a.slice[s] = ChainSlice{q.dst, (long long)q.dst_row_stride, q.out_offset, q.in_offset, q.pre,
                            q.post, q.scale};
  }
  a.sigmoid = c->sigmoid;
  a.sigmoid_scale = c->sigmoid_scale;
  a.sigmoid_off = c->sigmoid_offset;
  // A workgroup stores its rows while others still read theirs (one alone has read all of
  // its before it stores any).
  if (a.M > kChainRows) {
    const void *in = a.in ? (const void *)a.in : (const void *)a.in_f32;
    const long long size = (long long)a.M * a.K * (a.in ? 1 : 4), n = (long long)c->layers[a.layers - 1].N;
    bool touches = (a.out && rows_touch(a.out, n, a.M, n, in, size)) ||
                   (a.sigmoid && rows_touch(a.sigmoid, 4 * n, a.M, 4 * n, in, size));
    for (int s = 0; s < a.slices; s++)
      touches = touches || rows_touch(a.slice[s].dst, a.slice[s].pitch, a.M, n, in, size);
    MI355X_REQUIRE(!touches, "a destination overlaps the input of %d rows", a.M);
  }
  constexpr int W = 16;
  hipLaunchKernelGGL(fc_chain_i8_kernel<W>, dim3((a.M + kChainRows - 1) / kChainRows), dim3(W * 64), 0,
                     as_stream(stream), a);
  return check_launch("rwq_fc_chain_i8");
}
