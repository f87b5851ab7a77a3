// Decode attention of the float32 path, from the q|k|v projection: one kernel rotates a step's single tokens, stores their keys
// and values into the pages and attends, in 32-bit operands, products and sums throughout.
//
// A block is four waves on one (request, kv head), or on one of its key ranges (grid x): the group's G query heads share every
// key and value.  A wave takes every fourth tile of 16 keys, which lie in one page.  Scores: four lanes to a key, a quarter
// of the features each, in interleaved pieces of 16 bytes.  Values, stored [feature][slot], are read a lane to a feature; the
// weights reach all lanes through the wave's own patch of LDS, and each lane adds them up itself.  The next tile is fetched
// while this one is multiplied, and the first while the projection's pieces are on their way.  The new token's key and value
// go into the tile from LDS, so nobody waits for their stores.  The waves' states meet in LDS, in wave order; ranges are
// merged by merge_key_ranges_kernel.
//
// Bound by its chain of fetches (lengths and page ids, keys; beside them the projection) at short contexts and by the keys
// and values at long ones, which the general kernel read once per head.  32 heads on 8 kv heads of 64, us, before
// (rotation and general kernel) and now: 8 requests of 70 keys 13.6 -> 10.1, of 600 27 -> 15.1, of 4,000 81 -> 34.5, one of 4,000
// 49 -> 24, 64 of 2,000 393 -> 85; heads of 128, 8 requests of 2,000 84 -> 34.
#include "common.h"

typedef float f32x4_t __attribute__((ext_vector_type(4)));

struct Float32Projection {
  const float* part;      // [splits][T][ncols]
  int splits;
  long part_stride;
  int ncols, q_col, k_col, v_col;
  const float* table;     // [T, HD]: cosines of the HD / 2 pair angles, then their sines; null: no rotation
  int write_kv;
};

template <int HD, int G>
__global__ __launch_bounds__(256) void attention_float32_decode_kernel(float* __restrict__ out, long out_stride, Float32Projection src,
                                                                       float* k_cache, float* v_cache, const int* __restrict__ block_table, int table_width,
                                                                       const int* __restrict__ q_start, const int* __restrict__ kv_len_of, int nh, int nkv,
                                                                       int page_size, float scale, int window, long num_pages, float* __restrict__ part) {
  constexpr int KP = HD / 16, VF = HD / 64;          // a lane's pieces of a key; its features of the values
  __shared__ __attribute__((aligned(16))) float qs[G][HD], knew[HD], vnew[HD];
  __shared__ __attribute__((aligned(16))) float ps[4][G][16];
  __shared__ float ms[4][G], ls[4][G], os[4][G][HD];
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int split = blockIdx.x, splits = gridDim.x, g = blockIdx.y, r = blockIdx.z;
  const int p = kv_len_of[r] - 1;
  const long row = q_start[r];
  const int* bt = block_table + (long)r * table_width;
  const int lo = window > 0 && p - window + 1 > 0 ? p - window + 1 : 0;
  const int first_tile = lo / 16, tiles = p / 16 - first_tile + 1, per = (tiles + splits - 1) / splits;
  const int t0 = first_tile + split * per, t1 = min(first_tile + tiles, t0 + per);
  const bool newest = t0 < t1 && t1 == first_tile + tiles;         // the range ends at the new token

  const int key = lane / 4, quarter = lane % 4;
  f32x4_t kq[KP], vq[VF][4], kn[KP], vn[VF][4];
  auto page_of = [&](const int tile) -> long {
    const int blk = tile * 16 / page_size;
    const long page = blk < table_width ? bt[blk] : -1;
    return page < num_pages ? page : -1;
  };
  auto fetch = [&](const int tile, const long page, f32x4_t (&k)[KP], f32x4_t (&v)[VF][4]) {
    const long at = (page < 0 ? 0 : page) * nkv + g;               // a page that is not there: the first one, unused
    const int slot = tile * 16 % page_size;
    const float* kr = k_cache + (at * page_size + slot + key) * HD + quarter * 4;
    const float* vr = v_cache + at * page_size * HD + slot;
#pragma unroll
    for (int i = 0; i < KP; ++i) k[i] = *reinterpret_cast<const f32x4_t*>(kr + i * 16);
#pragma unroll
    for (int f = 0; f < VF; ++f)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[f][i] = *reinterpret_cast<const f32x4_t*>(vr + (long)(f * 64 + lane) * page_size + i * 4);
  };
  int tile = t0 + wave;
  long page = tile < t1 ? page_of(tile) : -1;
  if (tile < t1) fetch(tile, page, kq, vq);

  // the projection: pairs of the group's query heads, and where the range holds the new token of its key, then its values
  constexpr int Q_PAIRS = G * HD / 2, K_PAIRS = HD / 2;
  const int jobs = Q_PAIRS + (newest && src.write_kv ? K_PAIRS + HD : 0);
  const int new_blk = p / page_size, new_slot = p % page_size;
  const long new_page = newest && src.write_kv && new_blk < table_width ? bt[new_blk] : -1;
  const bool stored = new_page >= 0 && new_page < num_pages;       // the host checks tables; never write outside the pool
  const float* base = src.part + row * src.ncols;
  for (int job = tid; job < jobs; job += 256) {
    if (job >= Q_PAIRS + K_PAIRS) {
      const int d = job - Q_PAIRS - K_PAIRS;
      const float v = split_sum(base, src.splits, src.part_stride, src.v_col + g * HD + d);
      vnew[d] = v;
      if (stored) v_cache[((new_page * nkv + g) * HD + d) * page_size + new_slot] = v;
      continue;
    }
    const bool is_key = job >= Q_PAIRS;
    const int head = is_key ? 0 : job / (HD / 2), j = job % (HD / 2);
    const int col = is_key ? src.k_col + g * HD : src.q_col + (g * G + head) * HD;
    const float a = split_sum(base, src.splits, src.part_stride, col + j), b = split_sum(base, src.splits, src.part_stride, col + j + HD / 2);
    float x = a, y = b;
    if (src.table) rope_pair(a, b, src.table[row * HD + j], src.table[row * HD + HD / 2 + j], x, y);
    float* to = is_key ? knew : qs[head];
    to[j] = x;
    to[j + HD / 2] = y;
    if (is_key && stored) {
      float* kd = k_cache + ((new_page * nkv + g) * page_size + new_slot) * HD;
      kd[j] = x;
      kd[j + HD / 2] = y;
    }
  }
  __syncthreads();

  float m[G], l[G], acc[G][VF];
#pragma unroll
  for (int h = 0; h < G; ++h) {
    m[h] = -INFINITY;
    l[h] = 0.f;
#pragma unroll
    for (int f = 0; f < VF; ++f) acc[h][f] = 0.f;
  }
  const bool patch = newest && src.write_kv;
  while (tile < t1) {
    const int next = tile + 4;
    const long next_page = next < t1 ? page_of(next) : -1;
    if (next < t1) fetch(next, next_page, kn, vn);
    const int at = tile * 16;
    if (at < lo || at + 15 >= p) {                   // the first tile of a window, or the last: not all keys are seen
      if (patch && at + key == p) {
#pragma unroll
        for (int i = 0; i < KP; ++i) kq[i] = *reinterpret_cast<const f32x4_t*>(knew + i * 16 + quarter * 4);
      }
#pragma unroll
      for (int f = 0; f < VF; ++f)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          if (at + i < lo || at + i > p) vq[f][i / 4][i % 4] = 0.f;      // zero times what is not finite would not be zero
          else if (patch && at + i == p) vq[f][i / 4][i % 4] = vnew[f * 64 + lane];
        }
    }
#pragma unroll
    for (int h = 0; h < G; ++h) {
      f32x4_t dot = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < KP; ++i) {
        const f32x4_t q = *reinterpret_cast<const f32x4_t*>(&qs[h][i * 16 + quarter * 4]);
#pragma unroll
        for (int e = 0; e < 4; ++e) dot[e] = fmaf(q[e], kq[i][e], dot[e]);
      }
      float s = (dot[0] + dot[1]) + (dot[2] + dot[3]);
      s += __shfl_xor(s, 1, PI_WAVE);
      s += __shfl_xor(s, 2, PI_WAVE);
      s = at + key < lo || at + key > p ? -INFINITY : page < 0 ? __builtin_nanf("") : s * scale;   // a key without a page: visible
      float top = s;
#pragma unroll
      for (int off = 4; off < 64; off <<= 1) top = fmaxf(top, __shfl_xor(top, off, PI_WAVE));
      const float m_new = fmaxf(m[h], top);
      const float corr = m[h] == -INFINITY ? 0.f : expf(m[h] - m_new);
      if (quarter == 0) ps[wave][h][key] = s == -INFINITY ? 0.f : expf(s - m_new);
      m[h] = m_new;
      l[h] *= corr;
#pragma unroll
      for (int f = 0; f < VF; ++f) acc[h][f] *= corr;
    }
    // the wave reads what its own lanes wrote: LDS serves one wave's accesses in order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int h = 0; h < G; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x4_t w = *reinterpret_cast<const f32x4_t*>(&ps[wave][h][i * 4]);
        l[h] += (w[0] + w[1]) + (w[2] + w[3]);
#pragma unroll
        for (int f = 0; f < VF; ++f)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[h][f] = fmaf(w[e], vq[f][i][e], acc[h][f]);
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    tile = next;
    page = next_page;
#pragma unroll
    for (int i = 0; i < KP; ++i) kq[i] = kn[i];
#pragma unroll
    for (int f = 0; f < VF; ++f)
#pragma unroll
      for (int i = 0; i < 4; ++i) vq[f][i] = vn[f][i];
  }
#pragma unroll
  for (int h = 0; h < G; ++h) {
    if (lane == 0) {
      ms[wave][h] = m[h];
      ls[wave][h] = l[h];
    }
#pragma unroll
    for (int f = 0; f < VF; ++f) os[wave][h][f * 64 + lane] = acc[h][f];
  }
  __syncthreads();
  for (int at = tid; at < G * HD; at += 256) {
    const int h = at / HD, d = at % HD, head = g * G + h;
    float top = -INFINITY, sum = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) top = fmaxf(top, ms[w][h]);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      // a wave without keys weighs nothing; a score that is not a number keeps its maximum out of fmaxf, not out of the sums
      const float weight = ms[w][h] == -INFINITY ? (ls[w][h] == 0.f ? 0.f : 1.f) : expf(ms[w][h] - top);
      sum = fmaf(weight, ls[w][h], sum);
      o = fmaf(weight, os[w][h][d], o);
    }
    if (splits == 1) {
      out[row * out_stride + (long)head * HD + d] = o * (1.0f / sum);
    } else {
      float* mine = part + ((row * nh + head) * splits + split) * (HD + 2);
      mine[d] = o;
      if (d == 0) {
        mine[HD] = top;
        mine[HD + 1] = sum;
      }
    }
  }
}

int pi_merge_key_ranges_float32(float* out, long out_stride, const float* part, int T, int nh, int hd, int splits, hipStream_t stream);

// Sizes that the kernel takes: heads of 64 or 128, 1, 2, 3, 4 or 8 of them to a kv head.
extern "C" int pi_attention_float32_decode_takes(int nh, int nkv, int hd) {
  if (nkv <= 0 || nh <= 0 || nh % nkv || (hd != 64 && hd != 128)) return 0;
  const int G = nh / nkv;
  return G <= 4 || G == 8;
}

// One token per request.  The projection: float32 [splits][rows of the step][ncols], columns [q heads | k heads | v heads];
// `ranges`: key ranges per request and kv head, whose partial results go through `ranges_part` (R * nh * ranges * (hd + 2) floats).
extern "C" int pi_attention_float32_decode(void* out, long out_stride, const void* part, int splits, int ncols, int T, const void* table, int write_kv,
                                           void* k_cache, void* v_cache, const int* block_table, int table_width, const int* q_start, const int* kv_len,
                                           int R, int nh, int nkv, int hd, int page_size, float scale, int window, long num_pages, int ranges,
                                           void* ranges_part, long ranges_elems, hipStream_t stream) {
  PI_REQUIRE(pi_attention_float32_decode_takes(nh, nkv, hd), "float32 decode attention: not for %d heads on %d of %d", nh, nkv, hd);
  PI_REQUIRE(R > 0 && R == T && R <= 65535 && nkv <= 65535, "float32 decode attention: one token per request, got %d tokens of %d", T, R);
  PI_REQUIRE(page_size >= 16 && page_size % 16 == 0 && table_width > 0 && num_pages > 0, "float32 decode attention: pages of %d tokens", page_size);
  PI_REQUIRE(splits >= 1 && ncols >= (nh + (write_kv ? 2 * nkv : 0)) * hd, "float32 decode attention: %d columns do not hold q, k, v", ncols);
  PI_REQUIRE(window >= 0 && ranges >= 1 && ranges <= 64, "float32 decode attention: window %d, %d ranges", window, ranges);
  PI_REQUIRE(((uintptr_t)k_cache % 16 == 0) && ((uintptr_t)v_cache % 16 == 0), "float32 decode attention: the cache must be 16-byte aligned");
  PI_REQUIRE(ranges == 1 || (ranges_part && ranges_elems >= (long)R * nh * ranges * (hd + 2)), "float32 decode attention: workspace too small for %d ranges", ranges);
  const Float32Projection src{(const float*)part, splits, (long)T * ncols, ncols, 0, nh * hd, (nh + nkv) * hd, (const float*)table, write_kv};
  const dim3 grid(ranges, nkv, R), block(256);
#define GO(H, GR) \
  hipLaunchKernelGGL((attention_float32_decode_kernel<H, GR>), grid, block, 0, stream, (float*)out, out_stride, src, (float*)k_cache, (float*)v_cache, \
                     block_table, table_width, q_start, kv_len, nh, nkv, page_size, scale, window, num_pages, (float*)ranges_part)
#define GROUP(H) \
  switch (nh / nkv) { \
    case 1: GO(H, 1); break; \
    case 2: GO(H, 2); break; \
    case 3: GO(H, 3); break; \
    case 4: GO(H, 4); break; \
    default: GO(H, 8); break; \
  }
  if (hd == 64) { GROUP(64) } else { GROUP(128) }
#undef GROUP
#undef GO
  if (pi_check_launch("attention_float32_decode")) return -1;
  return ranges == 1 ? 0 : pi_merge_key_ranges_float32((float*)out, out_stride, (const float*)ranges_part, R, nh, hd, ranges, stream);
}
